"""The reconstruction at contracted widths of 128 and more (coupled bases): the
tile and segment edges of its workgroups, rows off a 16-byte boundary, the RoPE
epilogue with tables off one, and two problems in one launch."""
import numpy as np
import pytest
import torch

from oracle import attention as oa
from oracle import rope as orope
from slimkv_amd.workloads import rope_tables
from tests.helpers import assert_close, neighbour_of_exact, to_np

pytestmark = pytest.mark.gpu

D, HKV = 128, 8


def _inputs(device, B, n, R, shift):
    """Latent rows and W starting `shift` elements past a 16-byte boundary."""
    gen = torch.Generator(device=device).manual_seed(R + n)

    def take(*shape):
        size = int(np.prod(shape))
        flat = torch.randn(size + shift, generator=gen, device=device).to(torch.bfloat16)
        return flat[shift:].view(*shape)
    lat, w = take(B, n, R), take(HKV * D, R)
    return lat, w / 16 if not shift else w, torch.randn(HKV * D, generator=gen, device=device).to(torch.bfloat16)


@pytest.mark.parametrize('R,B,n,shift', [(128, 1, 1, 0), (192, 2, 17, 0), (256, 1, 33, 4), (384, 3, 1100, 0),
                                         (512, 1, 40, 0), (512, 2, 1025, 4), (192, 1, 16, 4)])
def test_wide_reconstruction(device, R, B, n, shift):
    from slimkv_amd import kernels
    lat, w, bias = _inputs(device, B, n, R, shift)
    plain = kernels.reconstruct(lat, w, bias, kv_heads=HKV)
    exact = oa.reconstruct(to_np(lat)[:, None], to_np(w), to_np(bias), HKV, D, bf16_boundaries=False)
    rounded = oa.reconstruct(to_np(lat)[:, None], to_np(w), to_np(bias), HKV, D)
    terms = oa.reconstruct(np.abs(to_np(lat))[:, None], np.abs(to_np(w)), None, HKV, D, bf16_boundaries=False)
    neighbour_of_exact(to_np(plain).transpose(0, 2, 1, 3), exact, rounded, terms)

    # RoPE and scatter: the reference's bf16 steps on the rows rebuilt above,
    # the tables one float past a 16-byte boundary where the rows are too
    off = 1 if shift else 0
    tables = [torch.empty(2000 * D + off, device=device)[off:].view(2000, D) for _ in range(2)]
    for t, src in zip(tables, rope_tables(2000, D, 500000.0, device)):
        t.copy_(src)
    cos, sin = tables
    gen = torch.Generator(device=device).manual_seed(5)
    pos = torch.randint(0, 2000, (B, n), generator=gen, device=device)
    dst = torch.randperm(n + 3, generator=torch.Generator().manual_seed(3))[:n].to(device)
    out = torch.zeros(B, HKV, n + 3, D, dtype=torch.bfloat16, device=device).transpose(1, 2)
    kernels.reconstruct(lat, w, bias, kv_heads=HKV, out=out, dst_rows=dst, positions=pos, cos=cos, sin=sin)
    c, s, p = to_np(cos).astype(np.float32), to_np(sin).astype(np.float32), pos.cpu().numpy()
    x = to_np(plain).astype(np.float32)
    rot = np.stack([orope.rotate_bf16(x[b], c[p[b]][:, None], s[p[b]][:, None]) for b in range(B)])
    np.testing.assert_array_equal(to_np(out)[:, dst.cpu().numpy()], rot)
    untouched = np.setdiff1d(np.arange(n + 3), dst.cpu().numpy())
    assert (to_np(out)[:, untouched] == 0).all()


@pytest.mark.parametrize('rows', [(16, 16), (300, 40), (2100, 2100)])
def test_wide_pair_equals_single_launches(device, rows):
    from slimkv_amd import kernels
    problems = [dict(zip(('latent', 'weight', 'bias'), _inputs(device, 1, n, 256, 0)), kv_heads=HKV) for n in rows]
    for got, kw in zip(kernels.reconstruct_pair(*problems), problems):
        assert torch.equal(got, kernels.reconstruct(**kw))


@pytest.mark.parametrize('rank,per_head,B,sink,n,raw,current', [(256, False, 2, 4, 300, 0, 70), (128, False, 1, 1, 17, 33, 1),
                                                                (512, False, 1, 0, 16, 5, 64), (32, True, 3, 4, 65, 7, 0),
                                                                (384, False, 2, 0, 1, 0, 129)])
def test_rows_around_a_rebuilt_history(device, rank, per_head, B, sink, n, raw, current):
    """[sink | up(history) | raw | current] in one call: the rebuilt rows are
    reconstruct's bits, the others copies, from strided and offset parts."""
    from types import SimpleNamespace
    from slimkv_amd import kernels
    from slimkv_amd.memory import ReconstructionCache
    from slimkv_amd.workloads import block_diagonal
    gen = torch.Generator(device=device).manual_seed(rank + n)

    def rnd(*shape):
        return torch.randn(*shape, generator=gen, device=device).to(torch.bfloat16)
    R = HKV * rank if per_head else rank
    up = torch.nn.Linear(R, HKV * D, bias=True, device=device, dtype=torch.bfloat16).requires_grad_(False)
    if per_head:
        up.weight.copy_(block_diagonal([rnd(D, rank) for _ in range(HKV)]))
    parts = [rnd(B, HKV, sink + 3, D)[:, :, 3:] if sink else None, rnd(B, raw, HKV, D).transpose(1, 2) if raw else None,
             rnd(B, current, HKV, 2 * D)[..., D:].transpose(1, 2) if current else None]
    latent = rnd(B, 1, n, R)
    cache = ReconstructionCache(parts[0], latent, parts[1], None, None, HKV, D, 'k')
    attention = SimpleNamespace(beacon_k_up_proj=up, num_key_value_heads=HKV, head_dim=D)
    got = cache.materialize(attention, parts[2])
    rebuilt = kernels.reconstruct(latent[:, 0], up.weight, up.bias, kv_heads=HKV, block_diagonal=per_head)
    want = torch.cat([x for x in (parts[0], rebuilt.transpose(1, 2), parts[1], parts[2]) if x is not None], 2)
    assert torch.equal(got, want)
    if current:                     # rows off a 16-byte boundary are copied by torch: the same result
        shifted = torch.empty(parts[2].numel() + 1, dtype=torch.bfloat16, device=device)[1:].view(parts[2].shape)
        shifted.copy_(parts[2])
        assert torch.equal(cache.materialize(attention, shifted), want)


def test_forward_mode_reaches_the_rows_around_a_history(device):
    """The tangents of sink and current rows are carried into the whole set, as
    torch's copies of them carry it."""
    from types import SimpleNamespace
    from torch.autograd import forward_ad
    from slimkv_amd.memory import ReconstructionCache
    gen = torch.Generator(device=device).manual_seed(9)
    up = torch.nn.Linear(256, HKV * D, bias=False, device=device, dtype=torch.bfloat16).requires_grad_(False)
    sink, current, dsink, dcurrent = (torch.randn(1, HKV, n, D, generator=gen, device=device).to(torch.bfloat16)
                                      for n in (4, 7, 4, 7))
    latent = torch.randn(1, 1, 20, 256, generator=gen, device=device).to(torch.bfloat16)
    attention = SimpleNamespace(beacon_k_up_proj=up, num_key_value_heads=HKV, head_dim=D)
    plain = ReconstructionCache(sink, latent, None, None, None, HKV, D, 'k').materialize(attention, current)
    with forward_ad.dual_level():
        cache = ReconstructionCache(forward_ad.make_dual(sink, dsink), latent, None, None, None, HKV, D, 'k')
        got, tangent = forward_ad.unpack_dual(cache.materialize(attention, forward_ad.make_dual(current, dcurrent)))
    assert torch.equal(got, plain)
    assert torch.equal(tangent, torch.cat([dsink, torch.zeros_like(tangent[:, :, 4:24]), dcurrent], 2))


@pytest.mark.parametrize('repeats', [True, False])
@pytest.mark.parametrize('R,B,n', [(256, 1, 33), (256, 2, 2100), (128, 2, 700), (384, 1, 17), (512, 1, 40), (512, 2, 1100)])
def test_decode_over_rebuilt_rotated_keys(device, R, B, n, repeats):
    """The reconstruction decode on coupled bases with beacon positions: RoPE
    from prepared pairs (rows that repeat their first half and rows that do
    not) and from the tables give the same bits; against float64 attention over
    the rows that reconstruct writes; stage by stage as in one call, with a
    prologue stage that leaves the workspace alone."""
    import ctypes
    from slimkv_amd import _lib, kernels
    gen = torch.Generator(device=device).manual_seed(R + n)

    def rnd(*shape, std=1.0):
        return (torch.randn(*shape, generator=gen, device=device) * std).to(torch.bfloat16)
    Hq, raw = 32, 21
    q, raw_k, raw_v = rnd(B, 1, Hq, D), rnd(B, raw, HKV, D), rnd(B, raw, HKV, D)
    lk, lv = rnd(B, n, R), rnd(B, n, R)
    uk, uv = rnd(HKV * D, R, std=R ** -0.5), rnd(HKV * D, R, std=R ** -0.5)
    bk, bv = rnd(HKV * D, std=0.1), rnd(HKV * D, std=0.1)
    cos, sin = rope_tables(4000, D, 500000.0, device)
    if not repeats:
        cos, sin = (torch.cat([t[:, :64], t[:, 64:].roll(7, 0)], 1).contiguous() for t in (cos, sin))
    assert bool(kernels.prepare_rope_pairs(cos, sin)[1]) == repeats
    pos = torch.full((B, 1), 3333, dtype=torch.int64, device=device)
    beacons = torch.randint(0, 4000, (B, n), generator=gen, device=device)
    kw = dict(beacon_positions=beacons, up_k_bias=bk, up_v_bias=bv, q_positions=pos, cos=cos, sin=sin)
    out, lse = kernels.recon_decode(q, raw_k, raw_v, lk, lv, uk, uv, D ** -0.5, **kw)

    base, plain, plain_lse, keep = kernels._latent_args(
        q, raw_k, raw_v, lk, lv, uk, uv, D ** -0.5, bk, bv, False, False, pos, cos, sin, None, None, 0, 0, None, None,
        prepared_bases=False)
    a = _lib.ReconDecodeArgs(base, beacons.data_ptr(), n, None, 0, 0)
    size = _lib.lib().slimkv_recon_decode_workspace(ctypes.byref(a))
    ws = torch.full((size,), 7, dtype=torch.uint8, device=device)
    for stage in (_lib.STAGE_PROLOGUE, _lib.STAGE_ATTEND, _lib.STAGE_COMBINE):
        _lib.check(_lib.lib().slimkv_recon_decode_stages(ctypes.byref(a), stage, ws.data_ptr(), size,
                                                         _lib.stream_handle(device)))
        assert stage != _lib.STAGE_PROLOGUE or bool((ws == 7).all())
    assert torch.equal(out, plain) and torch.equal(lse, plain_lse)

    key = kernels.reconstruct(lk, uk, bk, kv_heads=HKV, positions=beacons, cos=cos, sin=sin).double()
    value = kernels.reconstruct(lv, uv, bv, kv_heads=HKV).double()
    c, s = cos.to(torch.bfloat16).double()[3333], sin.to(torch.bfloat16).double()[3333]
    x = q[:, 0].double()
    x = (x * c + torch.cat([-x[..., 64:], x[..., :64]], -1) * s).view(B, HKV, Hq // HKV, D)
    key, value = (torch.cat([t, u.double()], 1).transpose(1, 2) for t, u in ((key, raw_k), (value, raw_v)))
    sc = x @ key.transpose(-1, -2).contiguous() * D ** -0.5
    assert_close(to_np(out[:, 0]), (torch.softmax(sc, -1) @ value.contiguous()).reshape(B, Hq, D).cpu().numpy(),
                 what=f'width {R}')


def test_rows_outside_the_output_are_refused(device):
    from slimkv_amd import kernels
    lat = torch.zeros(1, 20, 256, dtype=torch.bfloat16, device=device)
    w = torch.zeros(HKV * D, 256, dtype=torch.bfloat16, device=device)
    out = torch.zeros(1, HKV, 24, D, dtype=torch.bfloat16, device=device)
    part = torch.ones(1, HKV, 4, D, dtype=torch.bfloat16, device=device)
    kernels.reconstruct_with_rows(lat, w, None, out, 4, [(0, part)])
    for first, rows, weight, target in ((5, 0, w, out), (-1, 0, w, out), (4, 21, w, out), (4, -1, w, out),
                                        (4, 0, w[:, :128], out), (4, 0, w, out[..., :64]),
                                        (4, 0, w, out.expand(2, -1, -1, -1))):
        with pytest.raises(ValueError):
            kernels.reconstruct_with_rows(lat, weight, None, target, first, [(rows, part)])
    assert bool((out[:, :, :4] == 1).all()) and bool((out[:, :, 4:] == 0).all())
