"""Latent decode on coupled up-projections (every query head against whole
latent rows): the merge of the split partials and, below, sizes at the edges of
the kernels' tiles.  Against float64 attention over the rebuilt rows under the
parity bars of tests/helpers.py."""
import pytest
import torch

from slimkv_amd.workloads import rope_tables
from tests.helpers import MAX_ABS, assert_close, assert_lse_close, to_np

pytestmark = pytest.mark.gpu

D = 128


def _rope(x, cos, sin, pos):
    """float64 rotation by the tables' bf16 values."""
    c, s = cos.to(torch.bfloat16).double()[pos], sin.to(torch.bfloat16).double()[pos]
    return x * c + torch.cat([-x[..., D // 2:], x[..., :D // 2]], -1) * s


def layer(device, B, Hq, Hkv, n, raw, rk, rv, queries=1, bias=False, seed=0, capacity=None, lengths=None):
    """(call arguments, keywords, float64 output [B, L, Hq, D], LSE [B, Hq, L],
    LSE tolerance) of one layer; with `capacity` the rows sit in longer buffers
    of NaN with per-sequence lengths.

    The tolerance: an LSE is off by no more than the scores that dominate it,
    and a beacon's score is a sum over rotated query elements q_d k_d and, once
    absorbed, over q'_r l_r, each factor rounded to bf16 (relative error up to
    2^-9, the rotation's steps up to twice that).  Independent roundings add in
    squares, so a score's standard deviation is below 2^-9 times
    sqrt(sum (q_d k_d)^2 + sum (q'_r l_r)^2) times the scale; five of those for
    the largest one over all rows."""
    gen = torch.Generator(device=device).manual_seed(seed + n)

    def rnd(*shape, std=1.0):
        return (torch.randn(*shape, generator=gen, device=device) * std).to(torch.bfloat16)
    q, rk_rows, rv_rows = rnd(B, queries, Hq, D, std=2.0), rnd(B, raw, Hkv, D), rnd(B, raw, Hkv, D)
    lk, lv = rnd(B, n, rk), rnd(B, n, rv)
    uk, uv = rnd(Hkv * D, rk, std=rk ** -0.5), rnd(Hkv * D, rv, std=rv ** -0.5)
    bk, bv = (rnd(Hkv * D, std=0.1), rnd(Hkv * D, std=0.1)) if bias else (None, None)
    cos, sin = rope_tables(n + raw + 4, D, 500000.0, device)
    pos = (n + raw + torch.arange(queries, device=device))[None].expand(B, -1).contiguous()
    lens = [n] * B if lengths is None else lengths
    out = torch.empty(B, queries, Hq, D, dtype=torch.float64, device=device)
    lse = torch.empty(B, Hq, queries, dtype=torch.float64, device=device)
    G, noise = Hq // Hkv, 0.0
    for b in range(B):
        key, value = lk[b, :lens[b]].double() @ uk.double().t(), lv[b, :lens[b]].double() @ uv.double().t()
        if bias:
            key, value = key + bk.double(), value + bv.double()
        for h in range(Hkv):
            cols = slice(h * D, (h + 1) * D)
            k = torch.cat([rk_rows[b, :, h].double(), key[:, cols]])
            v = torch.cat([rv_rows[b, :, h].double(), value[:, cols]])
            for g in range(G):
                qr = _rope(q[b, :, h * G + g].double(), cos, sin, pos[b])
                sc = qr @ k.t() * D ** -0.5
                absorbed = qr @ uk[cols].double()
                var = qr ** 2 @ (k ** 2).t()
                var[:, raw:] += absorbed ** 2 @ (lk[b, :lens[b]].double() ** 2).t()
                noise = max(noise, float(var.max()) ** 0.5 * D ** -0.5 * 2 ** -9)
                for i in range(queries):                   # the first query of two does not see the last beacon
                    if queries == 2 and i == 0 and lens[b]:
                        sc[i, -1] = float('-inf')
                out[b, :, h * G + g] = torch.softmax(sc, -1) @ v
                lse[b, h * G + g] = torch.logsumexp(sc, -1)
    kw = dict(up_k_bias=bk, up_v_bias=bv, lat_causal=queries == 2, q_positions=pos, cos=cos, sin=sin)
    if capacity is not None:
        wide = [torch.full((B, capacity, w), float('nan'), dtype=torch.bfloat16, device=device) for w in (rk, rv)]
        for t, src in zip(wide, (lk, lv)):
            for b in range(B):
                t[b, :lens[b]] = src[b, :lens[b]]
        lk, lv = wide
        kw['lat_lengths'] = torch.tensor(lens, dtype=torch.int32, device=device)
    return (q, rk_rows, rv_rows, lk, lv, uk, uv, D ** -0.5), kw, out, lse, max(2e-3, 5 * noise)


def check(case, what, max_abs=MAX_ABS, **more):
    from slimkv_amd import kernels
    args, kw, out, lse, atol = case
    got, got_lse = kernels.latent_decode(*args, **dict(kw, **more))
    assert_close(to_np(got), out.cpu().numpy(), max_abs=max_abs, what=what)
    assert_lse_close(to_np(got_lse), lse.cpu().numpy(), atol=atol, what=what)
    return got, got_lse


@pytest.mark.parametrize('rank,raw,raw_splits,lat_splits', [(256, 40, 1, 1), (200, 529, 33, 7), (384, 70, 5, 256)])
def test_merge_of_many_and_few_splits(device, rank, raw, raw_splits, lat_splits):
    check(layer(device, 2, 32, 8, 4200, raw, rank, rank, bias=True, seed=rank), f'rank {rank}', raw_splits=raw_splits,
          lat_splits=lat_splits)


@pytest.mark.parametrize('width,splits', [(384, 1), (200, 64), (384, 256)])
def test_plain_attention_merge(device, width, splits):
    from slimkv_amd import kernels
    gen = torch.Generator(device=device).manual_seed(width + splits)
    q, k, v = (torch.randn(2, n, 4, width, generator=gen, device=device).to(torch.bfloat16) for n in (1, 4096, 4096))
    out, lse = kernels.attention_forward(q, k, v, width ** -0.5, splits=splits)
    sc = (q.double().transpose(1, 2) @ k.double().transpose(1, 2).transpose(-1, -2)) * width ** -0.5
    assert_close(to_np(out.transpose(1, 2)), (torch.softmax(sc, -1) @ v.double().transpose(1, 2)).cpu().numpy(),
                 what=f'width {width}')
    assert_lse_close(to_np(lse), torch.logsumexp(sc, -1).cpu().numpy(), what=f'width {width}')


# (batch, heads, KV heads, beacons, raw, K rank, V rank, queries, bias): one
# key, tile edges, widths at and beside the 128-column steps, unequal ranks,
# groups of 16 query rows from one to more than a workgroup holds
SIZES = [(1, 32, 8, 1, 5, 256, 256, 1, False), (2, 32, 8, 63, 133, 128, 64, 1, True),
         (3, 32, 8, 65, 20, 264, 248, 2, False), (1, 40, 8, 4097, 261, 320, 200, 2, True),
         (5, 8, 8, 1000, 9, 8, 384, 1, False), (1, 28, 4, 700, 70, 136, 8, 2, True),
         (2, 96, 8, 333, 17, 384, 384, 1, False), (1, 64, 8, 129, 33, 64, 120, 2, False)]


# several blocks of 64 columns to a workgroup of the query absorption: two or
# three of five, all of three, with a last block of 8 and of 64 columns
SIZES += [(22, 32, 8, 40, 5, 320, 200, 1, True), (70, 8, 8, 30, 5, 136, 72, 2, True)]


@pytest.mark.parametrize('B,Hq,Hkv,n,raw,rk,rv,queries,bias', SIZES)
def test_sizes(device, B, Hq, Hkv, n, raw, rk, rv, queries, bias):
    check(layer(device, B, Hq, Hkv, n, raw, rk, rv, queries, bias), f'{n} beacons')


# either side of the rule that gives few query rows over narrow latents to the
# split kernel: sequences, query rows, width
@pytest.mark.parametrize('B,Hq,rk,rv,queries', [(15, 8, 64, 64, 1), (16, 8, 64, 56, 1), (16, 8, 40, 64, 2),
                                                (16, 16, 8, 64, 1), (16, 24, 64, 64, 1), (16, 8, 72, 64, 1)])
def test_narrow_latents_of_few_heads(device, B, Hq, rk, rv, queries):
    lengths = [0 if queries == 1 else 2] + [(37 * i) % 300 + 2 for i in range(1, B)]
    for case in (layer(device, B, Hq, 8, 301, 21, rk, rv, queries, True, capacity=320, lengths=lengths),
                 layer(device, B, Hq, 8, 130, 5, rk, rv, queries)):
        # a key of few elements lets one row take all of the mass, and the
        # output is then that value row: the bf16 result and the bf16
        # probabilities are each off by up to 2^-8 of it
        check(case, f'{B} of {Hq} heads', max_abs=max(MAX_ABS, 2.0 ** -7 * float(case[2].abs().max())))


@pytest.mark.parametrize('B,width', [(63, 128), (64, 128), (64, 256), (63, 256)])
def test_long_runs_of_few_heads(device, B, width):
    """Sixteen tiles of 64 rows a CU and eight query rows; one set of rows for
    every sequence."""
    from slimkv_amd import kernels
    cu = torch.cuda.get_device_properties(device).multi_processor_count
    n = 64 * 16 * cu // 64
    gen = torch.Generator(device=device).manual_seed(width + B)

    def rnd(*shape, std=1.0):
        return (torch.randn(*shape, generator=gen, device=device) * std).to(torch.bfloat16)
    q, raw_k, raw_v = rnd(B, 1, 8, D), rnd(1, 9, 1, D), rnd(1, 9, 1, D)
    lat_k, lat_v = rnd(1, n, width), rnd(1, n, width)
    up_k, up_v = rnd(D, width, std=width ** -0.5), rnd(D, width, std=width ** -0.5)
    wide = [x.expand(B, *x.shape[1:]) for x in (raw_k, raw_v, lat_k, lat_v)]
    out, lse = kernels.latent_decode(q, *wide, up_k, up_v, D ** -0.5)
    key = torch.cat([raw_k[0, :, 0].double(), lat_k[0].double() @ up_k.double().t()])
    value = torch.cat([raw_v[0, :, 0].double(), lat_v[0].double() @ up_v.double().t()])
    sc = q[:, 0].double() @ key.t() * D ** -0.5
    assert_close(to_np(out[:, 0]), (torch.softmax(sc, -1) @ value).cpu().numpy(), what=f'width {width}')
    # a score is a sum of D terms over an absorbed query rounded to bf16: with
    # unit variances its error stays below five standard deviations of 2^-9
    assert_lse_close(to_np(lse[:, :, 0]), torch.logsumexp(sc, -1).cpu().numpy(), atol=5 * 2.0 ** -9,
                     what=f'width {width}')


@pytest.mark.parametrize('queries', [1, 2])
def test_capacity_buffers_and_lengths(device, queries):
    """Rows past a sequence's length are NaN and must not reach its result;
    lengths from none to all of the buffer."""
    lengths = [0, 1, 64, 700, 1024] if queries == 1 else [2, 1, 64, 700, 1024]
    check(layer(device, 5, 32, 8, 1024, 37, 200, 256, queries, capacity=1200, lengths=lengths), 'lengths')


@pytest.mark.parametrize('first', [1, 64, 1023])
def test_two_segments_equal_joined_rows(device, first):
    from slimkv_amd import kernels
    args, kw, *_ = layer(device, 2, 32, 8, 1024, 37, 192, 256, 2, True)
    q, rk, rv, lk, lv, *rest = args
    joined = kernels.latent_decode(*args, **kw)
    parts = kernels.latent_decode(q, rk, rv, lk[:, :first].clone(), lv[:, :first].clone(), *rest, **kw,
                                  lat_k2=lk[:, first:].clone(), lat_v2=lv[:, first:].clone())
    assert all(torch.equal(x, y) for x, y in zip(parts, joined))


# rows either side of a whole number of tiles a split, with few raw workgroups
# (three at 70 rows: the splits leave them CUs, 253 of 256) and with many (they
# do not)
@pytest.mark.parametrize('B,raw,n', [(1, 70, 253 * 64), (1, 70, 253 * 64 + 1), (1, 70, 256 * 64 + 1), (9, 1000, 1793)])
def test_split_counts(device, B, raw, n):
    check(layer(device, B, 8, 8, n, raw, 64, 64), f'{n} beacons')


@pytest.mark.parametrize('splits', [1, 7, 66, 256])
def test_given_splits(device, splits):
    """4200 rows are 66 tiles: seven splits of ten tiles, 66 of one."""
    check(layer(device, 1, 32, 8, 4200, 20, 64, 200), f'{splits} splits', lat_splits=splits)


def test_workspace_of_more_beacons_serves_fewer(device):
    """One raw workgroup leaves all CUs but one: as many tiles of 64 rows take
    a split each, one tile more half as many splits, and its workspace still
    holds the partials of the smaller call."""
    import ctypes
    from slimkv_amd import _lib, kernels
    cu = torch.cuda.get_device_properties(device).multi_processor_count
    few, many = (layer(device, 1, 8, 8, tiles * 64, 5, 64, 64) for tiles in (cu - 1, cu))

    def query(case, lat_splits=0):
        return kernels.latent_decode_workspace_bytes(*case[0], lat_splits=lat_splits)
    assert query(few) == query(few, lat_splits=cu - 1) > query(many, lat_splits=cu // 2)
    size = query(many)
    args, kw, out, lse, atol = few
    a, got, got_lse, keep = kernels._latent_args(
        *args, None, None, False, False, kw['q_positions'], kw['cos'], kw['sin'], None, None, 0, 0, None, None)
    workspace = torch.empty(size, dtype=torch.uint8, device=device)
    _lib.check(_lib.lib().slimkv_latent_decode(ctypes.byref(a), workspace.data_ptr(), size, _lib.stream_handle(device)))
    assert_close(to_np(got), out.cpu().numpy(), what='workspace of more beacons')
    assert_lse_close(to_np(got_lse), lse.cpu().numpy(), atol=atol, what='workspace of more beacons')


def test_strided_and_shared_rows(device):
    """Row strides past the width and one set of rows for every sequence give
    the bits of contiguous copies."""
    from slimkv_amd import kernels
    args, kw, *_ = layer(device, 3, 32, 8, 700, 37, 200, 256, 1, True)
    q, rk, rv, lk, lv, *rest = args
    wide_k, wide_v = (torch.cat([t, torch.full_like(t[..., :24], float('nan'))], -1) for t in (lk, lv))
    want = kernels.latent_decode(*args, **kw)
    got = kernels.latent_decode(q, rk, rv, wide_k[..., :200], wide_v[..., :256], *rest, **kw)
    assert all(torch.equal(x, y) for x, y in zip(got, want))
    shared = kernels.latent_decode(q, rk, rv, lk[:1].expand(3, -1, -1), lv[:1].expand(3, -1, -1), *rest, **kw)
    copied = kernels.latent_decode(q, rk, rv, lk[:1].repeat(3, 1, 1), lv[:1].repeat(3, 1, 1), *rest, **kw)
    assert all(torch.equal(x, y) for x, y in zip(shared, copied))


@pytest.mark.parametrize('B,n,raw,lat_splits', [(16, 2000, 517, 0), (1, 17000, 1800, 256), (2, 700, 40, 3)])
def test_device_scratch_gives_the_bits_of_a_workspace(device, B, n, raw, lat_splits):
    """80 query rows of width 384: the allocation-free call plans the splits of
    the call with a workspace, up to the largest partials that a plan has."""
    import ctypes
    from slimkv_amd import _lib, kernels
    gen = torch.Generator(device=device).manual_seed(n)

    def rnd(*shape, std=1.0):
        return (torch.randn(*shape, generator=gen, device=device) * std).to(torch.bfloat16)
    args = (rnd(B, 2, 40, D), rnd(B, raw, 8, D), rnd(B, raw, 8, D), rnd(B, n, 384), rnd(B, n, 384),
            rnd(8 * D, 384, std=0.05), rnd(8 * D, 384, std=0.05), D ** -0.5)
    want, want_lse = kernels.latent_decode(*args, lat_causal=True, lat_splits=lat_splits)
    a, got, got_lse, keep = kernels._latent_args(*args, None, None, False, True, None, None, None, None, None, 0,
                                                 lat_splits, None, None)
    _lib.check(_lib.lib().slimkv_latent_decode_noalloc(ctypes.byref(a), _lib.stream_handle(device)))
    torch.cuda.synchronize()
    assert torch.equal(got, want) and torch.equal(got_lse, want_lse)


def _shifted(t, by):
    """The values of t, starting `by` elements past a 16-byte boundary."""
    flat = torch.empty(t.numel() + by, dtype=t.dtype, device=t.device)[by:].view(t.shape)
    return flat.copy_(t)


@pytest.mark.parametrize('rank', [64, 128, 256])
@pytest.mark.parametrize('per_head', [False, True])
def test_operands_off_a_16_byte_boundary_give_the_same_bits(device, per_head, rank):
    """Queries, U_K and the K bias may start anywhere: copied, or read
    narrowly."""
    from slimkv_amd import kernels
    from slimkv_amd.workloads import block_diagonal
    args, kw, *_ = layer(device, 2, 32, 8, 300, 21, rank, rank, bias=True)
    q, rk, rv, lk, lv, uk, uv, scale = args
    if per_head:
        r = rank // 8
        uk, uv = (block_diagonal([t[128 * h:128 * h + 128, :r] for h in range(8)]) for t in (uk, uv))
    kw['block_diagonal'] = per_head
    want = kernels.latent_decode(q, rk, rv, lk, lv, uk, uv, scale, prepared_bases=False, **kw)
    for moved in ('q', 'up_k', 'bias'):
        got = kernels.latent_decode(_shifted(q, 4) if moved == 'q' else q, rk, rv, lk, lv,
                                    _shifted(uk, 1) if moved == 'up_k' else uk, uv, scale, prepared_bases=False,
                                    **dict(kw, up_k_bias=_shifted(kw['up_k_bias'], 3) if moved == 'bias' else kw['up_k_bias']))
        assert all(torch.equal(x, y) for x, y in zip(got, want)), moved
    if per_head:
        want = kernels.latent_decode(q, rk, rv, lk, lv, uk, uv, scale, **kw)
        got = kernels.latent_decode(_shifted(q, 4), rk, rv, lk, lv, _shifted(uk, 1), uv, scale, **kw)
        assert all(torch.equal(x, y) for x, y in zip(got, want))
    if per_head and rank == 64:
        return                              # the rebuild takes multiples of 16
    odd = torch.empty(2, 1, 32, 132, dtype=q.dtype, device=device)[..., 4:].copy_(q)
    single = q.as_strided(q.shape, (q.stride(0), 3, *q.stride()[2:]))          # one query: its stride is not used
    recon = [kernels.recon_decode(x, rk, rv, lk, lv, uk, uv, scale, **kw) for x in (q, _shifted(q, 1), odd, single)]
    assert all(torch.equal(x, y) for other in recon[1:] for x, y in zip(other, recon[0]))


@pytest.mark.parametrize('queries,positions', [(1, True), (2, True), (2, False)])
def test_raw_rows_alone(device, queries, positions):
    """No beacons: the queries are rotated for the raw rows only."""
    from slimkv_amd import kernels
    args, kw, *_ = layer(device, 3, 40, 8, 8, 77, 64, 64, queries)
    q, rk, rv, _, _, uk, uv, scale = args
    cos, sin, pos = kw['cos'], kw['sin'], kw['q_positions']
    rope = dict(cos=cos, sin=sin, q_positions=pos)
    if not positions:
        rows = kernels.query_rope_rows(cos, sin, pos)
        rope = dict(cos=rows[0], sin=rows[1])
    empty = torch.empty(3, 0, 64, dtype=q.dtype, device=device)
    got, lse = kernels.latent_decode(q, rk, rv, empty, empty, uk, uv, scale, **rope)
    c, s = (t.to(torch.bfloat16).double()[pos][:, :, None] for t in (cos, sin))
    x = q.double()
    x = (x * c + torch.cat([-x[..., 64:], x[..., :64]], -1) * s).view(3, queries, 8, 5, D).permute(0, 2, 3, 1, 4)
    k, v = (t.double().permute(0, 2, 1, 3)[:, :, None] for t in (rk, rv))
    sc = torch.matmul(x, k.transpose(-1, -2).contiguous()) * scale
    want = torch.matmul(torch.softmax(sc, -1), v).permute(0, 3, 1, 2, 4).reshape(3, queries, 40, D)
    assert_close(to_np(got), want.cpu().numpy(), max_abs=max(MAX_ABS, 2.0 ** -7 * float(want.abs().max())), what='raw rows')
