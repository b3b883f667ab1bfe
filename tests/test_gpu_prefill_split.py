"""The key-split schedule of the prefill attention: equal runs of key tiles over
the CUs, items in one, two or more runs, merged in fp32.  Against the unsplit
call and float64."""
import ctypes

import pytest
import torch

from tests.helpers import assert_close, assert_lse_close, to_np

pytestmark = pytest.mark.gpu

D = 128


@pytest.mark.parametrize('B,Hq,Hkv,L,N,causal', [(1, 32, 8, 1280, 9220, True), (1, 32, 8, 1, 33000, True),
                                                 (3, 20, 4, 300, 18000, True), (1, 64, 8, 129, 8193, False),
                                                 (2, 16, 16, 1000, 20011, True)])
def test_split_schedule(device, B, Hq, Hkv, L, N, causal):
    from slimkv_amd import _lib, kernels
    gen = torch.Generator(device=device).manual_seed(L + N)
    q, k, v = (torch.randn(B, n, h, D, generator=gen, device=device).to(torch.bfloat16)
               for n, h in ((L, Hq), (N, Hkv), (N, Hkv)))
    k[:, N // 2:] *= 2                       # the maximum moves between runs
    out, lse = kernels.prefill_attention(q, k, v, D ** -0.5, causal=causal)
    plain, plain_lse = torch.empty_like(out), torch.empty_like(lse)
    a = _lib.PrefillAttentionArgs(q.data_ptr(), *q.stride()[:3], k.data_ptr(), *k.stride()[:3], v.data_ptr(),
                                  *v.stride()[:3], plain.data_ptr(), *plain.stride()[:3], plain_lse.data_ptr(), None,
                                  B, L, Hq, Hkv, N, D, D ** -0.5, int(causal))
    assert _lib.lib().slimkv_prefill_attention_workspace(ctypes.byref(a)) > 0
    _lib.check(_lib.lib().slimkv_prefill_attention(ctypes.byref(a), _lib.stream_handle(device)))
    # The probabilities are rounded to bf16 (2^-9 relative) against the running
    # maximum of their own run, so numerator and denominator of the two results
    # each carry their own roundings: |difference| <= 4 * 2^-9 * sum p |v|, and
    # the two bf16 results 2^-9 of their size each; the LSEs 2 * 2^-9.
    weight = kernels.prefill_attention(q, k, v.abs(), D ** -0.5, causal=causal)[0].float()
    diff = (out.float() - plain.float()).abs()
    assert bool((diff <= 2.0 ** -7 * weight + 2.0 ** -8 * plain.float().abs()).all())
    assert_lse_close(to_np(lse), to_np(plain_lse), atol=2.0 ** -8)
    for b, h, rows in ((0, 0, slice(0, L)), (B - 1, Hq - 1, slice(max(0, L - 130), L))):
        kk, vv = k[b, :, h // (Hq // Hkv)].double(), v[b, :, h // (Hq // Hkv)].double()
        sc = q[b, rows, h].double() @ kk.t() * D ** -0.5
        if causal:
            i = torch.arange(L, device=device)[rows]
            sc = sc.masked_fill(torch.arange(N, device=device)[None] > i[:, None] + N - L, float('-inf'))
        assert_close(to_np(out[b, rows, h]), (torch.softmax(sc, -1) @ vv).cpu().numpy(), what=f'head {h}')


@pytest.mark.parametrize('repeats', [True, False])
@pytest.mark.parametrize('B,Hq,Hkv,L,N', [(1, 32, 8, 1280, 9220), (3, 20, 4, 300, 18000)])
def test_split_over_the_kept_set_with_query_rope(device, B, Hq, Hkv, L, N, repeats):
    """The window attention as the package calls it: K and V views of a kept
    [B, Hkv, capacity, D] set, queries of a [B, Hq, L, D] projection rotated at
    their positions from prepared pairs, rows that repeat their first half and
    rows that do not."""
    from slimkv_amd import _lib, kernels
    from slimkv_amd.workloads import rope_tables
    gen = torch.Generator(device=device).manual_seed(L + N)

    def rnd(*shape):
        return torch.randn(*shape, generator=gen, device=device).to(torch.bfloat16)
    q = rnd(B, Hq, L, D).transpose(1, 2)
    k, v = (rnd(B, Hkv, N + 700, D)[:, :, :N].transpose(1, 2) for _ in range(2))
    cos, sin = rope_tables(N + 50, D, 500000.0, device)
    if not repeats:
        cos, sin = (torch.cat([t[:, :64], t[:, 64:].roll(7, 0)], 1).contiguous() for t in (cos, sin))
    pos = (torch.arange(L, device=device) + N - L + 37)[None].expand(B, -1)
    out, lse = kernels.prefill_attention(q, k, v, D ** -0.5, q_positions=pos, cos=cos, sin=sin)
    pairs, same = kernels.prepare_rope_pairs(cos, sin)
    assert bool(same) == repeats
    plain, plain_lse = torch.empty_like(out), torch.empty_like(lse)
    a = _lib.PrefillAttentionArgs(q.data_ptr(), *q.stride()[:3], k.data_ptr(), *k.stride()[:3], v.data_ptr(),
                                  *v.stride()[:3], plain.data_ptr(), *plain.stride()[:3], plain_lse.data_ptr(), None,
                                  B, L, Hq, Hkv, N, D, D ** -0.5, 1, pairs.data_ptr(), pairs.shape[0], int(same),
                                  pos.data_ptr(), pos.stride(0))
    assert _lib.lib().slimkv_prefill_attention_workspace(ctypes.byref(a)) > 0
    _lib.check(_lib.lib().slimkv_prefill_attention(ctypes.byref(a), _lib.stream_handle(device)))
    # as above: both results round their probabilities against other maxima
    weight = kernels.prefill_attention(q, k, v.abs(), D ** -0.5, q_positions=pos, cos=cos, sin=sin)[0].float()
    diff = (out.float() - plain.float()).abs()
    assert bool((diff <= 2.0 ** -7 * weight + 2.0 ** -8 * plain.float().abs()).all())
    assert_lse_close(to_np(lse), to_np(plain_lse), atol=2.0 ** -8)
    c, s = (t.to(torch.bfloat16).double()[pos[0]] for t in (cos, sin))
    for b, h in ((0, 0), (B - 1, Hq - 1)):
        x = q[b, :, h].double()
        x = x * c + torch.cat([-x[:, 64:], x[:, :64]], 1) * s
        sc = x @ k[b, :, h // (Hq // Hkv)].double().t() * D ** -0.5
        i = torch.arange(L, device=device)
        sc = sc.masked_fill(torch.arange(N, device=device)[None] > i[:, None] + N - L, float('-inf'))
        assert_close(to_np(out[b, :, h]), (torch.softmax(sc, -1) @ v[b, :, h // (Hq // Hkv)].double()).cpu().numpy(),
                     what=f'head {h}')


def test_short_and_ragged_calls_run_whole(device):
    """No split where the runs would be short, the items fill the CUs evenly
    enough, or the key counts are known on the device only."""
    from slimkv_amd import _lib
    def plan(B, Hq, L, N, seqlens=None):
        a = _lib.PrefillAttentionArgs()
        a.batch, a.heads, a.kv_heads, a.queries, a.keys, a.head_dim, a.causal = B, Hq, Hq, L, N, D, 1
        a.seqlens_k = seqlens
        return _lib.lib().slimkv_prefill_attention_workspace(ctypes.byref(a))
    assert plan(1, 32, 1280, 9220) > 0
    assert plan(2, 40, 651, 911) == 0 and plan(4, 32, 1280, 9220) == 0 and plan(1, 32, 1280, 9220, 4096) == 0
    assert plan(1, 32, 1280, 1000) == 0 and plan(2, 32, 1024, 5024) == 0 and plan(1, 40, 300, 6300) > 0
