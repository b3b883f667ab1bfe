"""The general merge of split partials at the row and split counts where its
workgroup size changes (two and four rows a CU, 128 and 256 splits, many
partials of few rows), with and without the lift of a latent accumulator.
Against float64 attention over the same rows under the parity bars of
tests/helpers.py."""
import pytest
import torch

from tests.helpers import assert_close, assert_lse_close, to_np

pytestmark = pytest.mark.gpu

D = 128


def _rows_and_splits(device, case):
    cu = torch.cuda.get_device_properties(device).multi_processor_count
    return {'two a CU': (2 * cu, 3), 'more': (2 * cu + 1, 3), 'four a CU': (4 * cu, 2), 'many': (4 * cu + 1, 2),
            '128 splits': (3, 127), '129 splits': (4 * cu + 1, 129), '256 splits': (2, 256)}[case]


CASES = ['two a CU', 'more', 'four a CU', 'many', '128 splits', '129 splits', '256 splits']


@pytest.mark.parametrize('case', CASES)
def test_full_width_rows(device, case):
    from slimkv_amd import kernels
    rows, splits = _rows_and_splits(device, case)
    gen = torch.Generator(device=device).manual_seed(splits)
    W, n = 264, 16 * splits - 5
    q = torch.randn(rows, 1, 1, W, generator=gen, device=device).to(torch.bfloat16)
    k, v = (torch.randn(1, n, 1, W, generator=gen, device=device).to(torch.bfloat16) for _ in range(2))
    out, lse = kernels.attention_forward(q, k.expand(rows, -1, -1, -1), v.expand(rows, -1, -1, -1), W ** -0.5,
                                         splits=splits)
    sc = q[:, 0, 0].double() @ k[0, :, 0].double().t() * W ** -0.5
    assert_close(to_np(out[:, 0, 0]), (torch.softmax(sc, -1) @ v[0, :, 0].double()).cpu().numpy(), what=case)
    assert_lse_close(to_np(lse[:, 0, 0]), torch.logsumexp(sc, -1).cpu().numpy(), what=case)


@pytest.mark.parametrize('width', [72, 384])
@pytest.mark.parametrize('case', CASES)
def test_lifted_latents(device, case, width):
    """One KV head a sequence; the raw rows are one split of the counts above."""
    from slimkv_amd import kernels
    rows, splits = _rows_and_splits(device, case)
    gen = torch.Generator(device=device).manual_seed(width + splits)

    def rnd(*shape, std=1.0):
        return (torch.randn(*shape, generator=gen, device=device) * std).to(torch.bfloat16)
    n = 64 * (splits - 1) - 5
    q, raw_k, raw_v = rnd(rows, 1, 1, D), rnd(1, 9, 1, D), rnd(1, 9, 1, D)
    lat_k, lat_v = rnd(1, n, width), rnd(1, n, width)
    up_k, up_v = rnd(D, width, std=width ** -0.5), rnd(D, width, std=width ** -0.5)
    bias = rnd(D, std=0.1)
    out, lse = kernels.latent_decode(q, raw_k.expand(rows, -1, -1, -1), raw_v.expand(rows, -1, -1, -1),
                                     lat_k.expand(rows, -1, -1), lat_v.expand(rows, -1, -1), up_k, up_v, D ** -0.5,
                                     up_v_bias=bias, raw_splits=1, lat_splits=splits - 1)
    key = torch.cat([raw_k[0, :, 0].double(), lat_k[0].double() @ up_k.double().t()])
    value = torch.cat([raw_v[0, :, 0].double(), lat_v[0].double() @ up_v.double().t() + bias.double()])
    sc = q[:, 0, 0].double() @ key.t() * D ** -0.5
    assert_close(to_np(out[:, 0, 0]), (torch.softmax(sc, -1) @ value).cpu().numpy(), what=case)
    # a score is a sum of D terms over an absorbed query rounded to bf16: with
    # unit variances its error stays below five standard deviations of 2^-9
    assert_lse_close(to_np(lse[:, 0, 0]), torch.logsumexp(sc, -1).cpu().numpy(), atol=5 * 2.0 ** -9, what=case)
