// Split-K decode attention over coupled latents: every query head of a
// sequence against whole latent rows (up-projections that couple the KV
// heads), beside the raw rows of the same launch.  Included by attention.hip.
//
// A workgroup of eight waves owns (sequence, key split) with all query rows of
// the sequence, 16 PT of them, so each latent byte is read and staged once for
// every head; the split kernel's waves take eight query rows each and read the
// rows once per wave straight into MFMA lanes, where the cache's line lookups
// (sixteen rows per sixteen lanes) hold them back.  Per tile of 64 keys:
//   * the tile's K and V rows go to LDS in lane order from registers loaded a
//     tile ahead (64 KB in flight a CU at width 256);
//   * scores: wave (pg, kg) multiplies key tiles of 16 with the query rows of
//     one 16-row group it holds in registers, S^T[key, p], 16x16x32 MFMA;
//   * the waves' maxima meet in LDS, so all keep one online-softmax reference
//     per query row, and the probabilities go to LDS;
//   * O^T[v, p]: each wave owns 16 KQ value columns for all query rows, V^T
//     read from the row-major tile with transposing LDS reads.
// One workgroup a CU: a split's partials (rows x value width, fp32) are
// written once per workgroup instead of once per wave.
//
// Eight sequences of 8192 rows of width 256, 32 heads: 35.9 -> 23.7 us; three
// of 5461 rows (widths 320 and 200) with 80 query rows: 47.2 -> 19.0; one of
// 5003: 14.5 -> 9.8.  A tile takes 2.3 us of the first (7.3 TB/s over the
// chip); the rest is the launch, the first tile's round trip (5.6 us until it
// is in LDS) and the CUs that also hold raw workgroups, whose tiles come 4 us
// late.  Measured without gain: two workgroups a CU (24.5), raw workgroups
// last (25.5), raw splits of 16 rows (23.5).
#pragma once

namespace slimkv {

constexpr int kCoupledWaves = 8;
constexpr int kCoupledThreads = 64 * kCoupledWaves;
constexpr int kTileKeys = 64;

struct CoupledRows {
    const uint16_t* p; int64_t sb, sn;                // rows [0, n1)
    const uint16_t* p2; int64_t sb2, sn2;             // rows [n1, n), row i at index i - n1
    int width;
};

struct CoupledParams {
    const uint16_t* q;                                // absorbed query rows [B][Lq][Hq][k.width]
    CoupledRows k, v;
    int n1, n;
    const int32_t* seqlens;                           // keys of each sequence (<= n) or null
    int causal, splits, groups;                       // groups: workgroups that share the query rows
    float* part_ml;                                   // [B][Hq * Lq][splits][2]
    float* part_acc;                                  // [B][Hq * Lq][splits][v.width]
    int B, Lq, Hq, nwg;
    float scale_log2;
};

// KQ: width / 128, rounded up; PT: groups of 16 query rows.
template <int KQ, int PT>
struct CoupledShape {
    static constexpr int PG = PT <= 2 ? 2 : (PT <= 4 ? 4 : 8);   // waves that split the query rows
    static constexpr int KG = kCoupledWaves / PG;                // waves that split a tile's keys
    static constexpr int KG_USED = KG < 4 ? KG : 4;
    static constexpr int KT = kTileKeys / 16 / KG_USED;          // key tiles a wave
    static constexpr int KS = 4 * KQ;                            // k-steps of 32
    // A row's stride is an odd multiple of 32 bytes: eight rows' 16-byte
    // operand reads and four rows' 32-byte transposed reads meet distinct banks.
    static constexpr int STRIDE = 256 * KQ + 32;
    static constexpr int PSTRIDE = 2 * kTileKeys + 16;
    static constexpr int V_OFF = kTileKeys * STRIDE;
    static constexpr int P_OFF = 2 * V_OFF;
    static constexpr int MAX_OFF = P_OFF + 16 * PT * PSTRIDE;
    static constexpr int BYTES = MAX_OFF + KG * 16 * PT * 4;
    static constexpr int RAW_BYTES = kCoupledWaves * 2 * 16 * SplitLds<8>::RS * 2;
    static constexpr int LDS = BYTES > RAW_BYTES ? BYTES : RAW_BYTES;
};

// Four keys of one value column a lane from a row-major LDS tile: within each
// 16 lanes, lane l names row l / 4, columns 4 (l % 4) + [0, 4) and receives
// column l of the four rows.
typedef __attribute__((address_space(3))) v4s lds_v4s;
__device__ __forceinline__ v4s read_transposed(const char* p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(p));
}

template <int KQ, int PT>
__device__ __forceinline__ void coupled_body(const CoupledParams& prm, int w, char* lds) {
    using S = CoupledShape<KQ, PT>;
    constexpr int KS = S::KS, NP = 2 * KQ;            // NP: 16-byte pieces a thread stages of K, and of V
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, grp = lane >> 4;
    const int pg = wave % S::PG, kg = wave / S::PG;
    const int group = w % prm.groups;
    const int s = (w / prm.groups) % prm.splits;
    const int b = w / (prm.groups * prm.splits);
    const int P = prm.Lq * prm.Hq;
    const int p_first = group * 16 * PT;

    int Nb = prm.n;
    if (prm.seqlens) {
        const int sl = prm.seqlens[b];
        Nb = sl < 0 ? 0 : (sl < prm.n ? sl : prm.n);
    }
    // Tiles dealt round-robin over the splits, whatever the sequence's length:
    // the workgroups resident at one time read one window of its rows.
    const int tiles = (Nb + kTileKeys - 1) / kTileKeys;

    // The 16-byte pieces a thread stages of a tile, C a row for K and V alike:
    // piece i is row prow[i % PER] + i / PER * PSTEP, column pcol[i % PER] (512
    // pieces are whole rows of 16 or 32, 1536 of 48).  Columns past a width are
    // not staged; their loads repeat the row's first piece.
    constexpr int C = 16 * KQ, PER = KQ == 3 ? 3 : 1, PSTEP = PER * kCoupledThreads / C;
    const int ck = prm.k.width / 8, cv = prm.v.width / 8;
    int prow[PER], pcol[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        prow[i] = (kCoupledThreads * i + tid) / C;
        pcol[i] = (kCoupledThreads * i + tid) % C;
    }
    const uint16_t* k1 = prm.k.p + (int64_t)b * prm.k.sb;
    const uint16_t* v1 = prm.v.p + (int64_t)b * prm.v.sb;
    const uint16_t* k2 = prm.k.p2 + (int64_t)b * prm.k.sb2;
    const uint16_t* v2 = prm.v.p2 + (int64_t)b * prm.v.sb2;
    u32x4 ks_[NP], vs_[NP];
    auto row_of = [&](const uint16_t* a, int64_t sa, const uint16_t* c, int64_t sc, int r) {
        return r < prm.n1 ? a + (int64_t)r * sa : c + (int64_t)(r - prm.n1) * sc;
    };
    // Non-temporal loads up to width 256 (sixteen sequences of 8192 rows of
    // width 256: 55 against 60 us a layer), plain ones above, where rows end
    // inside cache lines more often (widths 320 and 200: 48 against 51 us).
    constexpr bool NT = KQ <= 2;
    auto fetch = [&](int t) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int r = min(t * kTileKeys + prow[i % PER] + i / PER * PSTEP, prm.n - 1), c = pcol[i % PER];
            ks_[i] = tile_load<NT>(row_of(k1, prm.k.sn, k2, prm.k.sn2, r) + (c < ck ? 8 * c : 0));
            vs_[i] = tile_load<NT>(row_of(v1, prm.v.sn, v2, prm.v.sn2, r) + (c < cv ? 8 * c : 0));
        }
    };
    if (s < tiles) fetch(s);

    // The wave's query rows (B operand: lane (p = col, grp) holds elements
    // 32 ks + 8 grp + [0, 8)), zero past the rows and the width.
    u32x4 qv[KS];
    const int pq = p_first + 16 * pg + col;
    {
        const bool ok = pg < PT && pq < P;
        const int j = ok ? pq / prm.Lq : 0, l = ok ? pq % prm.Lq : 0;
        const uint16_t* qrow = prm.q + (((int64_t)b * prm.Lq + l) * prm.Hq + j) * prm.k.width;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int k = 32 * ks + 8 * grp;
            const bool in = ok && k < prm.k.width;
            qv[ks] = zero_unless(in, *reinterpret_cast<const u32x4*>(qrow + (in ? k : 0)));
        }
    }
    const int lim = prm.causal ? Nb - prm.Lq + pq % prm.Lq + 1 : Nb;
    // Columns between the K width and the last k-step meet zero query
    // elements; zeroed once so that nothing non-finite is left there.
    for (int i = tid; i < kTileKeys * (16 * KQ - ck); i += kCoupledThreads) {
        const int r = i / (16 * KQ - ck), c = ck + i % (16 * KQ - ck);
        *reinterpret_cast<u32x4*>(lds + r * S::STRIDE + 16 * c) = u32x4{0u, 0u, 0u, 0u};
    }

    float m[PT], lsum = 0.f;
    v4f acc[KQ][PT];
#pragma unroll
    for (int t = 0; t < PT; ++t) {
        m[t] = kNegInf;
#pragma unroll
        for (int u = 0; u < KQ; ++u) acc[u][t] = v4f{0.f, 0.f, 0.f, 0.f};
    }
    float* smax = reinterpret_cast<float*>(lds + S::MAX_OFF);

    for (int t = s; t < tiles; t += prm.splits) {
        const int r0 = t * kTileKeys;
        // Rows past the sequence hold some other row: their scores are masked,
        // their values zeroed here (0 times a non-finite value).
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int row = prow[i % PER] + i / PER * PSTEP, c = pcol[i % PER];
            char* dst = lds + row * S::STRIDE + 16 * c;
            if (c < ck) *reinterpret_cast<u32x4*>(dst) = ks_[i];
            if (c < cv) *reinterpret_cast<u32x4*>(dst + S::V_OFF) = zero_unless(r0 + row < Nb, vs_[i]);
        }
        __syncthreads();
        if (t + prm.splits < tiles) fetch(t + prm.splits);

        // scores of the wave's keys and query rows
        float sv[S::KT][4];
        float tmax = kNegInf;
        if (pg < PT && kg < S::KG_USED) {
#pragma unroll
            for (int kt = 0; kt < S::KT; ++kt) {
                const int key = 16 * (kg * S::KT + kt);
                const char* krows = lds + (key + col) * S::STRIDE + 16 * grp;
                v4f sc0 = {0.f, 0.f, 0.f, 0.f}, sc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < KS; ks += 2) {
                    sc0 = mfma32(*reinterpret_cast<const u32x4*>(krows + 64 * ks), qv[ks], sc0);
                    sc1 = mfma32(*reinterpret_cast<const u32x4*>(krows + 64 * ks + 64), qv[ks + 1], sc1);
                }
                const v4f sc = sc0 + sc1;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    sv[kt][i] = r0 + key + 4 * grp + i < lim ? sc[i] : kNegInf;
                    tmax = fmaxf(tmax, sv[kt][i]);
                }
            }
            tmax = rows_max(tmax);
            if (grp == 0) smax[kg * 16 * PT + 16 * pg + col] = tmax;
        }
        __syncthreads();

        // one reference a query row for all waves
        float alpha[PT], mref_own = 0.f, alpha_own = 1.f;
#pragma unroll
        for (int i = 0; i < PT; ++i) {
            float x = smax[16 * i + col];
#pragma unroll
            for (int g2 = 1; g2 < S::KG_USED; ++g2) x = fmaxf(x, smax[g2 * 16 * PT + 16 * i + col]);
            const float mnew = fmaxf(m[i], x * prm.scale_log2);
            const float mref = mnew == kNegInf ? 0.f : mnew;
            alpha[i] = fast_exp2(m[i] - mref);
            m[i] = mnew;
            if (i == pg) {
                mref_own = mref;
                alpha_own = alpha[i];
            }
        }
        if (pg < PT && kg < S::KG_USED) {
            lsum *= alpha_own;
#pragma unroll
            for (int kt = 0; kt < S::KT; ++kt) {
                float p[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    p[i] = fast_exp2(fmaf(sv[kt][i], prm.scale_log2, -mref_own));
                    lsum += p[i];
                }
                *reinterpret_cast<u32x2*>(lds + S::P_OFF + (16 * pg + col) * S::PSTRIDE +
                                          2 * (16 * (kg * S::KT + kt) + 4 * grp)) =
                    u32x2{pack_bf16(p[0], p[1]), pack_bf16(p[2], p[3])};
            }
        }
        __syncthreads();

        // O^T[v, p] over the tile's keys
#pragma unroll
        for (int u = 0; u < KQ; ++u)
#pragma unroll
            for (int i = 0; i < PT; ++i) acc[u][i] *= alpha[i];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            u32x4 pb[PT];
#pragma unroll
            for (int i = 0; i < PT; ++i)
                pb[i] = *reinterpret_cast<const u32x4*>(lds + S::P_OFF + (16 * i + col) * S::PSTRIDE + 64 * h + 16 * grp);
#pragma unroll
            for (int u = 0; u < KQ; ++u) {
                const int v0 = 16 * (wave * KQ + u);
                if (v0 < prm.v.width) {
                    const char* src = lds + S::V_OFF + (32 * h + 8 * grp + (col >> 2)) * S::STRIDE + 2 * (v0 + 4 * (col & 3));
                    const u32x2 lo = __builtin_bit_cast(u32x2, read_transposed(src));
                    const u32x2 hi = __builtin_bit_cast(u32x2, read_transposed(src + 4 * S::STRIDE));
                    const u32x4 a = {lo.x, lo.y, hi.x, hi.y};
#pragma unroll
                    for (int i = 0; i < PT; ++i) acc[u][i] = mfma32(a, pb[i], acc[u][i]);
                }
            }
        }
        __syncthreads();
    }

    // masses: over a wave's lane groups, then over the waves that split the keys
    lsum = rows_sum(lsum);
    if (pg < PT && kg < S::KG_USED && grp == 0) smax[kg * 16 * PT + 16 * pg + col] = lsum;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PT; ++i) {
        const int p = p_first + 16 * i + col;
        if (p >= P) continue;
        const int64_t slot = ((int64_t)b * P + p) * prm.splits + s;
        if (wave == 0 && grp == 0) {
            float l = smax[16 * i + col];
#pragma unroll
            for (int g2 = 1; g2 < S::KG_USED; ++g2) l += smax[g2 * 16 * PT + 16 * i + col];
            prm.part_ml[2 * slot] = m[i];
            prm.part_ml[2 * slot + 1] = l;
        }
#pragma unroll
        for (int u = 0; u < KQ; ++u) {
            const int v = 16 * (wave * KQ + u) + 4 * grp;
            if (v < prm.v.width)
                *reinterpret_cast<v4f*>(prm.part_acc + slot * prm.v.width + v) = acc[u][i];
        }
    }
}

// Raw rows (split_segment, eight wave items a workgroup) come first in the
// grid, so that they drain while the latent workgroups stream.
template <int KQ, int PT>
__global__ void __launch_bounds__(kCoupledThreads) __attribute__((amdgpu_waves_per_eu(2)))
coupled_kernel(CoupledParams prm, Seg raw) {
    __shared__ __attribute__((aligned(16))) char lds[CoupledShape<KQ, PT>::LDS];
    const int w = blockIdx.x;
    if (w < raw.nwg) {
        split_segment<8, 1, 0, 0, 0, 0, kCoupledWaves>(raw, w, prm.B, prm.Lq, prm.Hq, prm.scale_log2, lds);
        return;
    }
    coupled_body<KQ, PT>(prm, w - raw.nwg, lds);
}

template <int KQ>
hipError_t launch_coupled_width(int pt, const CoupledParams& prm, const Seg& raw, hipStream_t st) {
    const dim3 grid(prm.nwg + raw.nwg), block(kCoupledThreads);
    switch (pt) {
        case 2: hipLaunchKernelGGL((coupled_kernel<KQ, 2>), grid, block, 0, st, prm, raw); break;
        case 3: hipLaunchKernelGGL((coupled_kernel<KQ, 3>), grid, block, 0, st, prm, raw); break;
        case 4: hipLaunchKernelGGL((coupled_kernel<KQ, 4>), grid, block, 0, st, prm, raw); break;
        case 5: hipLaunchKernelGGL((coupled_kernel<KQ, 5>), grid, block, 0, st, prm, raw); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_coupled(int pt, const CoupledParams& prm, const Seg& raw, hipStream_t st) {
    const int width = prm.k.width > prm.v.width ? prm.k.width : prm.v.width;
    if (width <= 128) return launch_coupled_width<1>(pt, prm, raw, st);
    if (width <= 256) return launch_coupled_width<2>(pt, prm, raw, st);
    return launch_coupled_width<3>(pt, prm, raw, st);
}

}  // namespace slimkv
