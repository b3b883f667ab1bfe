"""Latent decode on coupled up-projections (every query head against whole
latent rows): the merge of the split partials and, below, sizes at the edges of
the kernels' tiles.  Against float64 attention over the rebuilt rows under the
parity bars of tests/helpers.py."""
import pytest
import torch

from slimkv_amd.workloads import rope_tables
from tests.helpers import assert_close, assert_lse_close, to_np

pytestmark = pytest.mark.gpu

D = 128


def _rope(x, cos, sin, pos):
    """float64 rotation by the tables' bf16 values."""
    c, s = cos.to(torch.bfloat16).double()[pos], sin.to(torch.bfloat16).double()[pos]
    return x * c + torch.cat([-x[..., D // 2:], x[..., :D // 2]], -1) * s


def layer(device, B, Hq, Hkv, n, raw, rk, rv, queries=1, bias=False, seed=0, capacity=None, lengths=None):
    """(call arguments, keywords, float64 output [B, L, Hq, D], LSE [B, Hq, L])
    of one layer; with `capacity` the rows sit in longer buffers of NaN with
    per-sequence lengths."""
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
    G = Hq // Hkv
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
    return (q, rk_rows, rv_rows, lk, lv, uk, uv, D ** -0.5), kw, out, lse


def check(case, what, **more):
    from slimkv_amd import kernels
    args, kw, out, lse = case
    got, got_lse = kernels.latent_decode(*args, **dict(kw, **more))
    assert_close(to_np(got), out.cpu().numpy(), what=what)
    assert_lse_close(to_np(got_lse), lse.cpu().numpy(), atol=1e-2, what=what)
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
