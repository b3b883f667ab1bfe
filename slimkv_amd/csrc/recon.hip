// Beacon reconstruction (up-projection) on MFMA, with the bias, an optional
// bf16-exact RoPE epilogue and an optional row scatter.
//
// out[b, dst(n), h, :] = rope?(bf16(latent[b, n, :] @ W[h*D:(h+1)*D, :]^T + bias))
//
// One wavefront computes a 16-row x 128-feature block of one KV head as
// C^T[o, n] = W[o, :] . latent[n, :] on v_mfma_f32_16x16x16_bf16: the A operand
// (W rows) and the B operand (latent rows) are both contiguous along the
// contraction, so neither needs a transpose, and lane (n, g) ends with features
// o = 16t + 4g + i of row n for t = 0..7 -- d and d + 64 sit in the same lane,
// so rotate-half RoPE is applied in registers before the 8-byte stores.

#include "common.hpp"

#include <algorithm>

namespace slimkv {

struct ReconParams {
    const uint16_t* latent; int64_t l_sb, l_sn;
    const uint16_t* w; const uint16_t* bias; int64_t w_ld;   // W [Hkv*D, R] row-major
    uint16_t* out; int64_t o_sb, o_sn, o_sh;
    const int64_t* dst_rows;                                  // [n] or null (identity)
    const float* cos; const float* sin; int64_t rope_rows;
    const int64_t* positions; int64_t pos_sb;                 // [B, n] or null
    const uint32_t* pairs; int repeats;                       // (bf16 cos | bf16 sin << 16) rows of the tables or null
    int B, n, R, Hkv, blockdiag, k_lo_step;                   // k_lo_step: per-head latent slice width
    int in16, out16;                                          // latent and W / output rows 16-byte aligned
    int tables16;                                             // RoPE tables 16-byte aligned
    int row_frags;                                            // 16-row groups a tile of the wide kernel
};

constexpr int kReconWaves = 4;

template <int KSTEPS>
__global__ void __launch_bounds__(kReconWaves * 64)
recon_kernel(ReconParams p) {
    constexpr int D = 128;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = lane & 15, grp = lane >> 4;
    const int tiles = (p.n + 16 * kReconWaves - 1) / (16 * kReconWaves);
    const int h = blockIdx.x % p.Hkv;
    const int rt = (blockIdx.x / p.Hkv) % tiles;
    const int b = blockIdx.x / (p.Hkv * tiles);
    const int row = (rt * kReconWaves + wave) * 16 + col;
    const bool rv = row < p.n;
    const int k_lo = p.blockdiag ? h * p.k_lo_step : 0;

    const uint16_t* lrow = p.latent + (int64_t)b * p.l_sb + (int64_t)(rv ? row : 0) * p.l_sn + k_lo;
    v4f acc[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
        const int k = 16 * ks + 4 * grp;
        u32x2 bl = *reinterpret_cast<const u32x2*>(lrow + k);
        if (!rv) bl = u32x2{0u, 0u};
        const v4s bop = as_v4s(bl.x, bl.y);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const uint16_t* wr = p.w + ((int64_t)h * D + 16 * t + col) * p.w_ld + k_lo + k;
            const u32x2 al = *reinterpret_cast<const u32x2*>(wr);
            acc[t] = mfma16(as_v4s(al.x, al.y), bop, acc[t]);
        }
    }
    if (!rv) return;
    // lane holds x[d] for d = 16t + 4*grp + i
    float x[8][4];
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int d = 16 * t + 4 * grp + i;
            float v = acc[t][i];
            if (p.bias) v += bf16_to_f32(p.bias[(int64_t)h * D + d]);
            x[t][i] = round_bf16_hw(v);
        }
    if (p.positions) {
        const int64_t pos = clamp_i64(p.positions[(int64_t)b * p.pos_sb + row], 0, p.rope_rows - 1);
        const float* cr = p.cos + pos * D;
        const float* sr = p.sin + pos * D;
        float y[8][4];
#pragma unroll
        for (int t = 0; t < 8; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int d = 16 * t + 4 * grp + i;
                const float partner = t < 4 ? -x[t + 4][i] : x[t - 4][i];
                y[t][i] = round_bf16_hw(round_bf16_hw(x[t][i] * round_bf16_hw(cr[d])) + round_bf16_hw(partner * round_bf16_hw(sr[d])));
            }
#pragma unroll
        for (int t = 0; t < 8; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) x[t][i] = y[t][i];
    }
    const int64_t dst = p.dst_rows ? p.dst_rows[row] : row;
    uint16_t* orow = p.out + (int64_t)b * p.o_sb + dst * p.o_sn + (int64_t)h * p.o_sh;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const uint32_t lo = pack_bf16(x[t][0], x[t][1]);
        const uint32_t hi = pack_bf16(x[t][2], x[t][3]);
        *reinterpret_cast<u32x2*>(orow + 16 * t + 4 * grp) = u32x2{lo, hi};
    }
}

// Streaming variant for narrow contractions (kw <= 64): the wavefront keeps its
// head's W tile (A operand, 128 x kw) in registers and walks 16-row tiles with
// the next tile's latent rows already in flight, so W is read once per
// wavefront instead of once per tile.  Same epilogue as recon_kernel, which
// stays for these widths with RoPE tables off a 16-byte boundary.
template <int KSTEPS>
__device__ __forceinline__ void recon_stream_body(const ReconParams& p, int segs, int block) {
    constexpr int D = 128;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = lane & 15, grp = lane >> 4;
    const int h = block % p.Hkv;
    const int seg = (block / p.Hkv) % segs;
    const int b = block / (p.Hkv * segs);
    const int tiles = (p.n + 15) / 16;
    const int stride = segs * kReconWaves;
    const int k_lo = p.blockdiag ? h * p.k_lo_step : 0;
    u32x2 wa[8][KSTEPS];
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks)
            wa[t][ks] = *reinterpret_cast<const u32x2*>(p.w + ((int64_t)h * D + 16 * t + col) * p.w_ld + k_lo + 16 * ks +
                                                        4 * grp);
    float bias[8][4];
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            bias[t][i] = p.bias ? bf16_to_f32(p.bias[(int64_t)h * D + 16 * t + 4 * grp + i]) : 0.f;
    const uint16_t* lbase = p.latent + (int64_t)b * p.l_sb + k_lo + 4 * grp;
    auto load_rows = [&](u32x2 (&lr)[KSTEPS], int tile) {
        const int row = min(tile * 16 + col, p.n - 1);
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) lr[ks] = *reinterpret_cast<const u32x2*>(lbase + (int64_t)row * p.l_sn + 16 * ks);
    };
    int tile = seg * kReconWaves + wave;
    if (tile >= tiles) return;
    u32x2 cur[KSTEPS], nxt[KSTEPS];
    load_rows(cur, tile);
    for (; tile < tiles; tile += stride) {
        const bool more = tile + stride < tiles;
        load_rows(nxt, more ? tile + stride : tile);
        v4f acc[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) {
            const v4s bop = as_v4s(cur[ks].x, cur[ks].y);
#pragma unroll
            for (int t = 0; t < 8; ++t) acc[t] = mfma16(as_v4s(wa[t][ks].x, wa[t][ks].y), bop, acc[t]);
        }
        const int row = tile * 16 + col;
        if (row < p.n) {
            float x[8][4];
#pragma unroll
            for (int t = 0; t < 8; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) x[t][i] = round_bf16_hw(p.bias ? acc[t][i] + bias[t][i] : acc[t][i]);
            if (p.positions) {
                const int64_t pos = clamp_i64(p.positions[(int64_t)b * p.pos_sb + row], 0, p.rope_rows - 1);
                const float* cr = p.cos + pos * D;
                const float* sr = p.sin + pos * D;
                float y[8][4];
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    const float4 c4 = *reinterpret_cast<const float4*>(cr + 16 * t + 4 * grp);
                    const float4 s4 = *reinterpret_cast<const float4*>(sr + 16 * t + 4 * grp);
                    const float cv[4] = {c4.x, c4.y, c4.z, c4.w}, sv[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float partner = t < 4 ? -x[t + 4][i] : x[t - 4][i];
                        y[t][i] = round_bf16_hw(round_bf16_hw(x[t][i] * round_bf16_hw(cv[i])) + round_bf16_hw(partner * round_bf16_hw(sv[i])));
                    }
                }
#pragma unroll
                for (int t = 0; t < 8; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[t][i] = y[t][i];
            }
            const int64_t dst = p.dst_rows ? p.dst_rows[row] : row;
            uint16_t* orow = p.out + (int64_t)b * p.o_sb + dst * p.o_sn + (int64_t)h * p.o_sh;
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const uint32_t lo = pack_bf16(x[t][0], x[t][1]);
                const uint32_t hi = pack_bf16(x[t][2], x[t][3]);
                *reinterpret_cast<u32x2*>(orow + 16 * t + 4 * grp) = u32x2{lo, hi};
            }
        }
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) cur[ks] = nxt[ks];
    }
}

template <int KSTEPS>
__global__ void __launch_bounds__(kReconWaves * 64)
recon_stream_kernel(ReconParams p, int segs) {
    recon_stream_body<KSTEPS>(p, segs, blockIdx.x);
}

// Two reconstructions of the same latent width in one launch (the K and the
// V rebuild of a window's beacons): the first `blocks0` workgroups run the
// first, the rest the second -- each the single kernel's workgroup, so the
// results are the single launches' bits.
template <int KSTEPS>
__global__ void __launch_bounds__(kReconWaves * 64)
recon_stream_pair_kernel(ReconParams p0, ReconParams p1, int segs0, int segs1, int blocks0) {
    if ((int)blockIdx.x < blocks0) recon_stream_body<KSTEPS>(p0, segs0, blockIdx.x);
    else recon_stream_body<KSTEPS>(p1, segs1, blockIdx.x - blocks0);
}

// Wide contractions (kw >= 128: up-projections that couple every KV head).  A
// workgroup owns a head's 128 features and walks tiles of 16 RT rows; wave w
// holds the W rows of its own 32 features over the whole contraction in
// registers (64 VGPRs at kw 256) and multiplies them with the tile's latent
// rows on the 16x16x32 MFMA.  W (once a workgroup) and the latent rows go
// through LDS: an operand read straight from memory touches sixteen rows per
// sixteen lanes, and the cache's line lookups bound the kernel (7936 rows of
// width 256 on 8 heads: 26.9 us that way against 12.4 with whole rows read in
// lane order, 69.5 with W also read again for every tile; two problems of 256
// rows: 39 us as two such launches, 5.0 as one of these; the write of the
// rebuilt rows alone takes 3).  16-byte chunk c of row r sits at chunk
// c ^ (r & 7) of its LDS row, so eight lanes that read one chunk of eight
// rows meet eight different bank groups.
//
// Without RoPE the wave's features are 32w + 8*grp + [0, 8) a lane: the two A
// operands interleave the rows in fours, so a lane stores 16 contiguous
// bytes.  With RoPE they are 16w and 64 + 16w + [0, 16), so d and d + 64 share
// a lane for the rotation.
// AL16: latent and W rows 16-byte aligned, else 8-byte loads.
template <bool AL16>
__device__ __forceinline__ u32x4 load_piece(const uint16_t* src) {
    if constexpr (AL16) {
        return *reinterpret_cast<const u32x4*>(src);
    } else {
        const u32x2 lo = *reinterpret_cast<const u32x2*>(src);
        const u32x2 hi = *reinterpret_cast<const u32x2*>(src + 4);
        return u32x4{lo.x, lo.y, hi.x, hi.y};
    }
}

// LDS of a workgroup: two tiles of 32 rows, or 16 W rows for each wave.
template <int KS>
struct WideLds {
    static constexpr int bytes = 2 * 32 * KS * 64;
};

template <int KS, int RT, bool ROPE, bool AL16>
__device__ __forceinline__ void recon_wide_body(const ReconParams& p, int segs, int block, char* lds) {
    constexpr int D = 128;
    constexpr int C = 4 * KS;                 // 16-byte chunks of a row
    constexpr int ROWS = 16 * RT;
    constexpr int CHUNKS = ROWS * C;
    constexpr int PIECES = (CHUNKS + 255) / 256;   // chunks a thread stages of a tile
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = lane & 15, grp = lane >> 4;
    // Row segments fastest over the 8 XCDs (workgroups are dealt to them in
    // turn), heads next: an XCD's L2 then holds the rows of its segments for
    // every head.
    int h, seg;
    const int b = block / (p.Hkv * segs);
    const int rest = block % (p.Hkv * segs);
    if (segs % 8 == 0) {
        h = (rest / 8) % p.Hkv;
        seg = rest / (8 * p.Hkv) * 8 + rest % 8;
    } else {
        h = rest % p.Hkv;
        seg = rest / p.Hkv;
    }
    const int tiles = (p.n + ROWS - 1) / ROWS;
    const int k_lo = p.blockdiag ? h * p.k_lo_step : 0;
    auto feature = [&](int f, int r) { return ROPE ? 64 * f + 16 * wave + r : 32 * wave + 8 * (r >> 2) + 4 * f + (r & 3); };
    auto slot = [](int row, int chunk) { return (row * C + (chunk ^ (row & 7))) * 16; };

    int tile = seg;
    if (tile >= tiles) return;                // the whole workgroup
    const uint16_t* lbase = p.latent + (int64_t)b * p.l_sb + k_lo;
    u32x4 stage[PIECES];
    auto fetch = [&](int t) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            const int id = min(256 * i + (int)threadIdx.x, CHUNKS - 1);
            stage[i] = load_piece<AL16>(lbase + (int64_t)min(t * ROWS + id / C, p.n - 1) * p.l_sn + 8 * (id % C));
        }
    };
    auto put = [&](char* buf) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            const int id = 256 * i + threadIdx.x;
            if (CHUNKS % 256 == 0 || id < CHUNKS) *reinterpret_cast<u32x4*>(buf + slot(id / C, id % C)) = stage[i];
        }
    };
    auto operand = [&](const char* buf, int row, int ks) {
        return *reinterpret_cast<const u32x4*>(buf + slot(row, 4 * ks + grp));
    };

    // W: every load of both operands and of the first tile goes out at once;
    // then each wave stages the 16 rows of one operand at a time in its own
    // part of the LDS.
    u32x4 wa[2][KS];
    char* own = lds + wave * 16 * C * 16;
    {
        u32x4 w[2][C / 4];
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int i = 0; i < C / 4; ++i) {
                const int id = 64 * i + lane;
                w[f][i] = load_piece<AL16>(p.w + ((int64_t)h * D + feature(f, id / C)) * p.w_ld + k_lo + 8 * (id % C));
            }
        fetch(tile);
#pragma unroll
        for (int f = 0; f < 2; ++f) {
#pragma unroll
            for (int i = 0; i < C / 4; ++i) {
                const int id = 64 * i + lane;
                *reinterpret_cast<u32x4*>(own + slot(id / C, id % C)) = w[f][i];
            }
            __syncthreads();
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) wa[f][ks] = operand(own, col, ks);
            __syncthreads();
        }
    }
    float bias[2][4];
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int i = 0; i < 4; ++i) bias[f][i] = p.bias ? bf16_to_f32(p.bias[(int64_t)h * D + feature(f, 4 * grp + i)]) : 0.f;

    // A lane's (bf16 cos | bf16 sin << 16) pairs, loaded before the tile's
    // products: from prepared pairs one 16-byte piece serves both operands
    // where a row repeats its first half, from the fp32 tables four (K rotated
    // and V of 8192 rows of width 256: 32.6 us as two launches from the
    // tables, 27.3 as one from the pairs).
    struct RopePiece {
        u32x4 f[2];
    };
    auto load_rope = [&](RopePiece& t, int row) {
        const int64_t pos = clamp_i64(p.positions[(int64_t)b * p.pos_sb + min(row, p.n - 1)], 0, p.rope_rows - 1);
        if (p.pairs) {
            const uint32_t* pr = p.pairs + pos * D + 4 * grp;
            t.f[0] = *reinterpret_cast<const u32x4*>(pr + 16 * wave);
            t.f[1] = p.repeats ? t.f[0] : *reinterpret_cast<const u32x4*>(pr + 64 + 16 * wave);
            return;
        }
#pragma unroll
        for (int f = 0; f < 2; ++f) {
            const float* cr = p.cos + pos * D + feature(f, 4 * grp);
            const float* sr = p.sin + pos * D + feature(f, 4 * grp);
            float4 c, s;
            if (p.tables16) {
                c = *reinterpret_cast<const float4*>(cr);
                s = *reinterpret_cast<const float4*>(sr);
            } else {
                c = make_float4(cr[0], cr[1], cr[2], cr[3]);
                s = make_float4(sr[0], sr[1], sr[2], sr[3]);
            }
            t.f[f] = u32x4{pack_bf16(c.x, s.x), pack_bf16(c.y, s.y), pack_bf16(c.z, s.z), pack_bf16(c.w, s.w)};
        }
    };
    auto finish = [&](const v4f (&acc)[2], const RopePiece& t, int row) {
        if (row >= p.n) return;
        float x[2][4];
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int i = 0; i < 4; ++i) x[f][i] = round_bf16_hw(p.bias ? acc[f][i] + bias[f][i] : acc[f][i]);
        const int64_t dst = p.dst_rows ? p.dst_rows[row] : row;
        uint16_t* orow = p.out + (int64_t)b * p.o_sb + dst * p.o_sn + (int64_t)h * p.o_sh;
        if constexpr (ROPE) {
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                float y[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float partner = f == 0 ? -x[1][i] : x[0][i];
                    y[i] = round_bf16_hw(x[f][i] * lo_bf16(t.f[f][i])) + round_bf16_hw(partner * hi_bf16(t.f[f][i]));
                }
                *reinterpret_cast<u32x2*>(orow + feature(f, 4 * grp)) = u32x2{pack_bf16(y[0], y[1]), pack_bf16(y[2], y[3])};
            }
        } else {
            const u32x4 w = {pack_bf16(x[0][0], x[0][1]), pack_bf16(x[0][2], x[0][3]), pack_bf16(x[1][0], x[1][1]),
                             pack_bf16(x[1][2], x[1][3])};
            uint16_t* o = orow + 32 * wave + 8 * grp;
            if (p.out16) {
                *reinterpret_cast<u32x4*>(o) = w;
            } else {
                *reinterpret_cast<u32x2*>(o) = u32x2{w.x, w.y};
                *reinterpret_cast<u32x2*>(o + 4) = u32x2{w.z, w.w};
            }
        }
    };
    // Double-buffered tiles, one barrier a tile: a wave writes buffer `at`
    // only after the barrier that every wave reached past its reads of it.
    for (int at = 0; tile < tiles; tile += segs, at ^= 1) {
        char* buf = lds + at * 32 * C * 16;
        put(buf);
        __syncthreads();
        RopePiece rope[RT];
        if constexpr (ROPE) {
#pragma unroll
            for (int r = 0; r < RT; ++r) load_rope(rope[r], tile * ROWS + 16 * r + col);
        }
        if (tile + segs < tiles) fetch(tile + segs);
        v4f acc[RT][2];
#pragma unroll
        for (int r = 0; r < RT; ++r) acc[r][0] = acc[r][1] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                const u32x4 lr = operand(buf, 16 * r + col, ks);
#pragma unroll
                for (int f = 0; f < 2; ++f) acc[r][f] = mfma32(wa[f][ks], lr, acc[r][f]);
            }
#pragma unroll
        for (int r = 0; r < RT; ++r) finish(acc[r], rope[r], tile * ROWS + 16 * r + col);
    }
}

template <int KS, int RT, bool ROPE, bool AL16>
__global__ void __launch_bounds__(kReconWaves * 64) __attribute__((amdgpu_waves_per_eu(2)))
recon_wide_kernel(ReconParams p, int segs) {
    __shared__ __attribute__((aligned(16))) char lds[WideLds<KS>::bytes];
    recon_wide_body<KS, RT, ROPE, AL16>(p, segs, blockIdx.x, lds);
}

// Two reconstructions of one width in one launch, as recon_stream_pair_kernel.
template <int KS, int RT, bool ROPE>   // ROPE: of the first
__global__ void __launch_bounds__(kReconWaves * 64) __attribute__((amdgpu_waves_per_eu(2)))
recon_wide_pair_kernel(ReconParams p0, ReconParams p1, int segs0, int segs1, int blocks0) {
    __shared__ __attribute__((aligned(16))) char lds[WideLds<KS>::bytes];
    if ((int)blockIdx.x < blocks0) recon_wide_body<KS, RT, ROPE, true>(p0, segs0, blockIdx.x, lds);
    else recon_wide_body<KS, RT, false, true>(p1, segs1, blockIdx.x - blocks0, lds);
}

// Full-width rows beside the rebuilt ones ([sink | history | raw | current] of
// a history rebuild): copied by extra workgroups of the same launch, 64 rows
// each, sixteen lanes a 256-byte row.
struct RowCopies {
    static constexpr int kMax = 3;
    const uint16_t* src[kMax]; int64_t sb[kMax], sh[kMax], sn[kMax];
    int64_t dst_row[kMax];                                    // first row of the output
    int rows[kMax], groups[kMax];                             // rows of a head, workgroups (0: no such copy)
    int count;
};
constexpr int kCopyRows = 64;

__device__ __forceinline__ void copy_rows(const RowCopies& c, const ReconParams& p, int block) {
    // One call per copy: an index into the kernel arguments, or a select
    // between their fields, would put them in scratch memory.
    auto copy = [&](const uint16_t* src, int64_t sb, int64_t sh, int64_t sn, int64_t dst_row, int rows, int at_block) {
        const int total = p.B * p.Hkv * rows;
        const int piece = 8 * (threadIdx.x & 15);
        u32x4 v[kCopyRows / 16];
        int64_t at[kCopyRows / 16];
#pragma unroll
        for (int u = 0; u < kCopyRows / 16; ++u) {
            // past the end: the last row again
            const int r = min(at_block * kCopyRows + 16 * u + (int)(threadIdx.x >> 4), total - 1);
            const int n = r % rows, h = r / rows % p.Hkv, b = r / rows / p.Hkv;
            v[u] = *reinterpret_cast<const u32x4*>(src + b * sb + h * sh + n * sn + piece);
            at[u] = b * p.o_sb + h * p.o_sh + (dst_row + n) * p.o_sn + piece;
        }
#pragma unroll
        for (int u = 0; u < kCopyRows / 16; ++u) *reinterpret_cast<u32x4*>(p.out + at[u]) = v[u];
    };
    if (block < c.groups[0]) {
        copy(c.src[0], c.sb[0], c.sh[0], c.sn[0], c.dst_row[0], c.rows[0], block);
        return;
    }
    block -= c.groups[0];
    if (block < c.groups[1]) {
        copy(c.src[1], c.sb[1], c.sh[1], c.sn[1], c.dst_row[1], c.rows[1], block);
        return;
    }
    copy(c.src[2], c.sb[2], c.sh[2], c.sn[2], c.dst_row[2], c.rows[2], block - c.groups[1]);
}

__global__ void __launch_bounds__(kReconWaves * 64) copy_rows_kernel(ReconParams p, RowCopies c) {
    copy_rows(c, p, blockIdx.x);
}

// `shift`: the copies' rows count from the output's first row, the rebuilt ones
// from p.out + shift.
template <int KS, int RT>
__global__ void __launch_bounds__(kReconWaves * 64) __attribute__((amdgpu_waves_per_eu(2)))
recon_wide_copies_kernel(ReconParams p, int segs, int blocks, int64_t shift, RowCopies c) {
    __shared__ __attribute__((aligned(16))) char lds[WideLds<KS>::bytes];
    if ((int)blockIdx.x >= blocks) {
        copy_rows(c, p, blockIdx.x - blocks);
        return;
    }
    p.out += shift;
    recon_wide_body<KS, RT, false, true>(p, segs, blockIdx.x, lds);
}

namespace {
bool al4(int64_t x) { return (x & 3) == 0; }
bool pal8(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 7) == 0; }
bool al8(int64_t x) { return (x & 7) == 0; }
bool pal16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }

template <int KS, int RT>
hipError_t launch_wide_rt(const ReconParams& p, int segs, hipStream_t st) {
    const dim3 grid(p.B * p.Hkv * segs), block(kReconWaves * 64);
    if (p.positions) {
        if constexpr (KS < 16 || RT == 1) {                // width 512 with RoPE has one row group (prepare_recon)
            if (p.in16) hipLaunchKernelGGL((recon_wide_kernel<KS, RT, true, true>), grid, block, 0, st, p, segs);
            else hipLaunchKernelGGL((recon_wide_kernel<KS, RT, true, false>), grid, block, 0, st, p, segs);
        }
    } else {
        if (p.in16) hipLaunchKernelGGL((recon_wide_kernel<KS, RT, false, true>), grid, block, 0, st, p, segs);
        else hipLaunchKernelGGL((recon_wide_kernel<KS, RT, false, false>), grid, block, 0, st, p, segs);
    }
    return hipGetLastError();
}

template <int KS>
hipError_t launch_wide(const ReconParams& p, int segs, hipStream_t st) {
    return p.row_frags == 1 ? launch_wide_rt<KS, 1>(p, segs, st) : launch_wide_rt<KS, 2>(p, segs, st);
}

template <int K>
hipError_t launch_recon(const ReconParams& p, int grid, hipStream_t st) {
    hipLaunchKernelGGL((recon_kernel<K>), dim3(grid), dim3(kReconWaves * 64), 0, st, p);
    return hipGetLastError();
}

template <int K>
hipError_t launch_stream(const ReconParams& p, int segs, hipStream_t st) {
    hipLaunchKernelGGL((recon_stream_kernel<K>), dim3(p.B * p.Hkv * segs), dim3(kReconWaves * 64), 0, st, p, segs);
    return hipGetLastError();
}
}  // namespace

// Workgroups of a wide reconstruction: each loads its head's W once, so few of
// them, but the CUs want more than one (7936 rows of width 256, K and V with
// the rows around them: 47 / 41 / 41 / 45 us at 256 / 512 / 768 / 1024).
constexpr int kWideGroups = 512;

// Checks a reconstruction and fills its kernel parameters; `segs` > 0 when it
// takes the streaming kernel (latent width kw <= 64) or the wide one
// (kw >= 128), whose workgroup count is B * Hkv * segs.
int prepare_recon(const slimkv_reconstruct_args* a, ReconParams* out, int* segs, int* kw_out) {
    if (!a) return fail(SLIMKV_EINVAL, "null pointer");
    if (a->batch <= 0 || a->rows < 0 || a->rank <= 0 || a->kv_heads <= 0 || a->head_dim != 128)
        return fail(SLIMKV_EINVAL, "invalid reconstruction sizes (head_dim must be 128)");
    *segs = 0;
    *kw_out = 0;
    if (a->rows == 0) return SLIMKV_OK;               // nothing to read or write (empty tensors may be null)
    if (!a->latent || !a->weight || !a->out) return fail(SLIMKV_EINVAL, "null pointer");
    const bool bd = a->block_diagonal != 0;
    const int64_t kw = bd ? a->rank / a->kv_heads : a->rank;
    if ((bd && a->rank % a->kv_heads) || kw % 16 || kw > 512)
        return fail(SLIMKV_EUNSUP, "the contracted latent width must be a multiple of 16 up to 512");
    const int64_t strides[] = {a->l_sb, a->l_sn, a->o_sb, a->o_sn, a->o_sh, a->rank};
    for (int64_t s : strides)
        if (!al4(s)) return fail(SLIMKV_EINVAL, "strides must be multiples of 4 elements");
    if (!pal8(a->latent) || !pal8(a->weight) || !pal8(a->out)) return fail(SLIMKV_EINVAL, "tensors must be 8-byte aligned");
    if (a->positions && (!a->cos || !a->sin || a->rope_rows <= 0)) return fail(SLIMKV_EINVAL, "RoPE needs tables");
    if (a->positions && a->batch > 1 && a->pos_sb < a->rows)
        return fail(SLIMKV_EINVAL, "positions rows are shorter than the row count");
    ReconParams& p = *out;
    p = ReconParams{};
    p.latent = static_cast<const uint16_t*>(a->latent); p.l_sb = a->l_sb; p.l_sn = a->l_sn;
    p.w = static_cast<const uint16_t*>(a->weight); p.bias = static_cast<const uint16_t*>(a->bias); p.w_ld = a->rank;
    p.out = static_cast<uint16_t*>(a->out); p.o_sb = a->o_sb; p.o_sn = a->o_sn; p.o_sh = a->o_sh;
    p.dst_rows = a->dst_rows;
    p.cos = a->cos; p.sin = a->sin; p.rope_rows = a->rope_rows;
    p.positions = a->positions; p.pos_sb = a->pos_sb;
    p.B = (int)a->batch; p.n = (int)a->rows; p.R = (int)a->rank; p.Hkv = (int)a->kv_heads;
    p.blockdiag = bd ? 1 : 0; p.k_lo_step = (int)kw;
    p.in16 = pal16(a->latent) && pal16(a->weight) && al8(a->l_sb) && al8(a->l_sn) && al8(a->rank);
    p.out16 = pal16(a->out) && al8(a->o_sb) && al8(a->o_sn) && al8(a->o_sh);
    *kw_out = (int)kw;
    p.tables16 = !a->positions || (((reinterpret_cast<uintptr_t>(a->cos) | reinterpret_cast<uintptr_t>(a->sin)) & 15) == 0);
    if (kw <= 64 && p.tables16) {
        // streaming kernel: about 1024 workgroups, each wavefront at least one tile
        const int row_tiles = (p.n + 15) / 16;
        const int64_t heads = (int64_t)p.B * p.Hkv;
        const int sg = (int)std::max<int64_t>(1, std::min<int64_t>((row_tiles + kReconWaves - 1) / kReconWaves,
                                                                   (1024 + heads - 1) / heads));
        if ((int64_t)p.B * p.Hkv * sg > 0x3fffffff) return fail(SLIMKV_EINVAL, "reconstruction grid too large");
        *segs = sg;
    } else if (kw >= 128) {
        // wide kernel: tiles of 32 rows, of 16 where 32 would leave CUs idle;
        // (and where W of width 512 and the RoPE pieces leave no registers for
        // the second group: it spilled); row segments in eights where there
        // are that many (its XCD order)
        const int64_t heads = (int64_t)p.B * p.Hkv;
        p.row_frags = heads * ((p.n + 31) / 32) < kWideGroups / 2 || (kw == 512 && a->positions) ? 1 : 2;
        const int row_tiles = (p.n + 16 * p.row_frags - 1) / (16 * p.row_frags);
        int sg = (int)std::max<int64_t>(1, std::min<int64_t>(row_tiles, (kWideGroups + heads - 1) / heads));
        if (sg >= 8) sg = sg / 8 * 8;
        if (heads * sg > 0x3fffffff) return fail(SLIMKV_EINVAL, "reconstruction grid too large");
        *segs = sg;
    }
    return SLIMKV_OK;
}

int launch_prepared(const ReconParams& p, int segs, int kw, hipStream_t st) {
    hipError_t e;
    if (segs > 0) {
        switch (kw / 16) {
            case 1: e = launch_stream<1>(p, segs, st); break;
            case 2: e = launch_stream<2>(p, segs, st); break;
            case 3: e = launch_stream<3>(p, segs, st); break;
            case 4: e = launch_stream<4>(p, segs, st); break;
            case 8: e = launch_wide<4>(p, segs, st); break;
            case 12: e = launch_wide<6>(p, segs, st); break;
            case 16: e = launch_wide<8>(p, segs, st); break;
            case 24: e = launch_wide<12>(p, segs, st); break;
            case 32: e = launch_wide<16>(p, segs, st); break;
            default: return fail(SLIMKV_EUNSUP, "latent width not instantiated");
        }
        return check_hip(e, "reconstruction kernel launch");
    }
    const int tiles = (p.n + 16 * kReconWaves - 1) / (16 * kReconWaves);
    const int grid = p.B * tiles * p.Hkv;
    switch (kw / 16) {
        case 1: e = launch_recon<1>(p, grid, st); break;
        case 2: e = launch_recon<2>(p, grid, st); break;
        case 3: e = launch_recon<3>(p, grid, st); break;
        case 4: e = launch_recon<4>(p, grid, st); break;
        default: return fail(SLIMKV_EUNSUP, "latent width not instantiated");
    }
    return check_hip(e, "reconstruction kernel launch");
}

template <int K>
hipError_t launch_stream_pair(const ReconParams& p0, int segs0, const ReconParams& p1, int segs1, hipStream_t st) {
    const int blocks0 = p0.B * p0.Hkv * segs0;
    const int blocks1 = p1.B * p1.Hkv * segs1;
    hipLaunchKernelGGL((recon_stream_pair_kernel<K>), dim3(blocks0 + blocks1), dim3(kReconWaves * 64), 0, st, p0, p1,
                       segs0, segs1, blocks0);
    return hipGetLastError();
}

template <int KS>
hipError_t launch_wide_pair(const ReconParams& p0, int segs0, const ReconParams& p1, int segs1, hipStream_t st) {
    const int blocks0 = p0.B * p0.Hkv * segs0;
    const int blocks1 = p1.B * p1.Hkv * segs1;
    const dim3 grid(blocks0 + blocks1), block(kReconWaves * 64);
#define SLIMKV_PAIR(RT, ROPE) \
    hipLaunchKernelGGL((recon_wide_pair_kernel<KS, RT, ROPE>), grid, block, 0, st, p0, p1, segs0, segs1, blocks0)
    if (p0.row_frags == 1) {
        if (p0.positions) SLIMKV_PAIR(1, true);
        else SLIMKV_PAIR(1, false);
    } else if (!p0.positions) {
        SLIMKV_PAIR(2, false);
    } else {
        if constexpr (KS < 16) SLIMKV_PAIR(2, true);       // width 512 with RoPE has one row group (prepare_recon)
    }
#undef SLIMKV_PAIR
    return hipGetLastError();
}

int reconstruct_pair(const slimkv_reconstruct_args* a, const slimkv_reconstruct_args* b, hipStream_t st,
                     const uint32_t* pairs, int repeats) {
    ReconParams pa{}, pb{};
    int sa = 0, sb = 0, ka = 0, kb = 0;
    int rc = prepare_recon(a, &pa, &sa, &ka);
    if (rc != SLIMKV_OK) return rc;
    if (pairs && pa.positions && pal16(pairs)) {
        pa.pairs = pairs;
        pa.repeats = repeats;
    }
    if (!b) return a->rows == 0 ? SLIMKV_OK : launch_prepared(pa, sa, ka, st);
    rc = prepare_recon(b, &pb, &sb, &kb);
    if (rc != SLIMKV_OK) return rc;
    if (a->rows == 0) return b->rows == 0 ? SLIMKV_OK : launch_prepared(pb, sb, kb, st);
    if (b->rows == 0) return launch_prepared(pa, sa, ka, st);
    // wide widths share a launch with 16-byte rows and RoPE at most of the first
    const bool pairable =
        ka <= 64 || (!pb.positions && pa.in16 && pb.in16 && pa.row_frags == pb.row_frags);
    if (sa > 0 && sb > 0 && ka == kb && pairable) {
        hipError_t e;
        switch (ka / 16) {
            case 1: e = launch_stream_pair<1>(pa, sa, pb, sb, st); break;
            case 2: e = launch_stream_pair<2>(pa, sa, pb, sb, st); break;
            case 3: e = launch_stream_pair<3>(pa, sa, pb, sb, st); break;
            case 4: e = launch_stream_pair<4>(pa, sa, pb, sb, st); break;
            case 8: e = launch_wide_pair<4>(pa, sa, pb, sb, st); break;
            case 12: e = launch_wide_pair<6>(pa, sa, pb, sb, st); break;
            case 16: e = launch_wide_pair<8>(pa, sa, pb, sb, st); break;
            case 24: e = launch_wide_pair<12>(pa, sa, pb, sb, st); break;
            case 32: e = launch_wide_pair<16>(pa, sa, pb, sb, st); break;
            default: return fail(SLIMKV_EUNSUP, "latent width not instantiated");
        }
        return check_hip(e, "reconstruction pair launch");
    }
    // different kernels or widths: two launches
    rc = launch_prepared(pa, sa, ka, st);
    return rc != SLIMKV_OK ? rc : launch_prepared(pb, sb, kb, st);
}

namespace {

template <int KS>
hipError_t launch_wide_copies(const ReconParams& p, int segs, int64_t shift, const RowCopies& c, int groups,
                              hipStream_t st) {
    const int blocks = p.B * p.Hkv * segs;
    const dim3 grid(blocks + groups), block(kReconWaves * 64);
    if (p.row_frags == 1)
        hipLaunchKernelGGL((recon_wide_copies_kernel<KS, 1>), grid, block, 0, st, p, segs, blocks, shift, c);
    else
        hipLaunchKernelGGL((recon_wide_copies_kernel<KS, 2>), grid, block, 0, st, p, segs, blocks, shift, c);
    return hipGetLastError();
}

}  // namespace

int reconstruct_with_rows(const slimkv_reconstruct_args* a, const slimkv_row_copy* copies, int count, hipStream_t st) {
    if (!a || count < 0 || count > RowCopies::kMax || (count && !copies)) return fail(SLIMKV_EINVAL, "invalid row copies");
    ReconParams p{};
    int segs = 0, kw = 0;
    int rc = prepare_recon(a, &p, &segs, &kw);
    if (rc != SLIMKV_OK) return rc;
    RowCopies c{};
    void* out = nullptr;
    int64_t groups = 0;
    for (int i = 0; i < count; ++i) {
        const slimkv_row_copy& r = copies[i];
        if (r.rows < 0 || r.first_row < 0 || a->batch * a->kv_heads * r.rows > (1 << 30))
            return fail(SLIMKV_EINVAL, "invalid row copy");
        if (r.rows == 0) continue;
        if (!r.src || !r.out || !pal16(r.src) || !pal16(r.out) || !al8(r.sb) || !al8(r.sn) || !al8(r.sh) ||
            !al8(a->o_sb) || !al8(a->o_sn) || !al8(a->o_sh))
            return fail(SLIMKV_EINVAL, "row copies need 16-byte aligned rows");
        if (c.count && r.out != out) return fail(SLIMKV_EINVAL, "row copies share one output");
        out = r.out;
        c.src[c.count] = static_cast<const uint16_t*>(r.src);
        c.sb[c.count] = r.sb; c.sh[c.count] = r.sh; c.sn[c.count] = r.sn;
        c.dst_row[c.count] = r.first_row;
        c.rows[c.count] = (int)r.rows;
        c.groups[c.count] = (int)((a->batch * a->kv_heads * r.rows + kCopyRows - 1) / kCopyRows);
        groups += c.groups[c.count++];
    }
    if (!c.count) return a->rows == 0 ? SLIMKV_OK : launch_prepared(p, segs, kw, st);
    ReconParams whole = p;
    if (a->rows == 0) {
        whole.B = (int)a->batch; whole.Hkv = (int)a->kv_heads;
        whole.o_sb = a->o_sb; whole.o_sn = a->o_sn; whole.o_sh = a->o_sh;
    }
    whole.out = static_cast<uint16_t*>(out);
    if (a->rows > 0 && kw >= 128 && !p.positions && p.in16 && p.out16) {
        const int64_t shift = p.out - whole.out;
        hipError_t e;
        switch (kw / 16) {
            case 8: e = launch_wide_copies<4>(whole, segs, shift, c, (int)groups, st); break;
            case 12: e = launch_wide_copies<6>(whole, segs, shift, c, (int)groups, st); break;
            case 16: e = launch_wide_copies<8>(whole, segs, shift, c, (int)groups, st); break;
            case 24: e = launch_wide_copies<12>(whole, segs, shift, c, (int)groups, st); break;
            case 32: e = launch_wide_copies<16>(whole, segs, shift, c, (int)groups, st); break;
            default: return fail(SLIMKV_EUNSUP, "latent width not instantiated");
        }
        return check_hip(e, "reconstruction kernel launch");
    }
    if (a->rows > 0) {
        rc = launch_prepared(p, segs, kw, st);
        if (rc != SLIMKV_OK) return rc;
    }
    hipLaunchKernelGGL(copy_rows_kernel, dim3((unsigned)groups), dim3(kReconWaves * 64), 0, st, whole, c);
    return check_hip(hipGetLastError(), "row copy launch");
}

}  // namespace slimkv

extern "C" int slimkv_reconstruct_with_rows(const slimkv_reconstruct_args* a, const slimkv_row_copy* copies,
                                            int32_t count, void* stream) {
    return slimkv::reconstruct_with_rows(a, copies, count, static_cast<hipStream_t>(stream));
}

extern "C" int slimkv_reconstruct(const slimkv_reconstruct_args* a, void* stream) {
    return slimkv::reconstruct_pair(a, nullptr, static_cast<hipStream_t>(stream));
}

extern "C" int slimkv_reconstruct_pair(const slimkv_reconstruct_args* a, const slimkv_reconstruct_args* b,
                                       void* stream) {
    return slimkv::reconstruct_pair(a, b, static_cast<hipStream_t>(stream));
}
