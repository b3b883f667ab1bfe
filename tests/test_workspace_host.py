"""Workspace queries (no GPU needed: nothing here launches a kernel): a size
asked for once serves the calls that the header says it serves."""
import ctypes

import pytest


def latent_args(batch, heads, beacons, rank_k, rank_v, *, queries=1, kv_heads=8, raw=133, raw_splits=0, lat_splits=0,
                per_head=False):
    from slimkv_amd import _lib
    a = _lib.LatentDecodeArgs()
    for name in ('q', 'raw_k', 'raw_v', 'lat_k', 'lat_v', 'up_k', 'up_v', 'out'):
        setattr(a, name, 1 << 20)           # any aligned address: a query reads no data
    a.batch, a.queries, a.heads, a.kv_heads, a.head_dim = batch, queries, heads, kv_heads, 128
    a.raw_keys, a.lat_keys, a.rank_k, a.rank_v, a.scale = raw, beacons, rank_k, rank_v, 128 ** -0.5
    a.raw_splits, a.lat_splits, a.block_diagonal = raw_splits, lat_splits, int(per_head)
    return a


def latent_workspace(*args, **kw):
    from slimkv_amd import _lib
    return _lib.lib().slimkv_latent_decode_workspace(ctypes.byref(latent_args(*args, **kw)))


@pytest.mark.parametrize('batch,heads,queries,rank', [(1, 8, 1, 64), (16, 8, 1, 64), (16, 8, 1, 128), (64, 8, 1, 256),
                                                      (1, 32, 1, 256), (8, 32, 1, 256), (3, 40, 2, 320),
                                                      (300, 32, 1, 128)])
def test_fewer_beacons_fit_the_workspace_of_more(batch, heads, queries, rank):
    """Bases without blocks, automatic splits."""
    sizes = [latent_workspace(batch, heads, n, rank, rank, queries=queries)
             for n in sorted({*range(1, 20000, 331), *(64 * t for t in range(250, 260)), 16384, 16385})]
    assert sizes[0] > 0 and sizes == sorted(sizes)


@pytest.mark.parametrize('rank', [128, 256])
@pytest.mark.parametrize('sequences', [8, 55, 56])
def test_a_larger_row_total_fits_the_workspace_of_a_smaller(sequences, rank):
    from slimkv_amd import _lib
    sizes = []
    for total in [65543, *range(704 * 256 - 900, 704 * 256 + 1200, 300), 704 * 256 - 1, 704 * 256, 1 << 18, 1 << 19]:
        a = _lib.PagedLatentDecodeArgs()
        a.base = latent_args(sequences, 32, 65536, rank, rank, per_head=True)
        a.base.lat_lengths = a.pages = a.table = 1 << 20
        a.slots, a.sink_elements, a.page_stride, a.num_pages = 4, 0, 8 * rank, 1 << 20
        a.t_cols = a.t_sb = 1 << 14
        a.rows_total = total
        sizes.append((total, _lib.lib().slimkv_paged_latent_decode_workspace(ctypes.byref(a))))
    sizes = [size for _, size in sorted(sizes)]
    assert sizes[-1] > 0 and sizes == sorted(sizes, reverse=True)


def test_device_scratch_constant_matches_the_header():
    import re
    from pathlib import Path
    from slimkv_amd import _lib
    header = (Path(__file__).resolve().parents[1] / 'include' / 'slimkv_hip.h').read_text()
    mib = int(re.search(r'SLIMKV_NOALLOC_SCRATCH_BYTES \((\d+)u << 20\)', header).group(1))
    assert _lib.NOALLOC_SCRATCH_BYTES == mib << 20


@pytest.mark.parametrize('batch,heads,queries', [(1, 40, 2), (3, 40, 2), (16, 40, 2), (51, 40, 2), (2, 96, 1),
                                                 (64, 32, 1), (128, 32, 2), (256, 8, 1)])
@pytest.mark.parametrize('rank_v', [256, 384])
def test_the_device_scratch_holds_coupled_partials(batch, heads, queries, rank_v):
    """The allocation-free call has a fixed scratch: with few raw rows it takes
    every coupled plan up to 256 sequences, whatever its beacons, and a given
    split count takes no more than it says."""
    from slimkv_amd import _lib
    for beacons in (64, 1000, 4096, 16384, 100000):
        assert 0 < latent_workspace(batch, heads, beacons, 384, rank_v, queries=queries, raw=64) <= _lib.NOALLOC_SCRATCH_BYTES
    for beacons in (130, 1000, 4200):
        given = [latent_workspace(batch, heads, beacons, 384, rank_v, queries=queries, lat_splits=n) for n in range(1, 40)]
        rows = batch * heads * queries
        for n, size in enumerate(given, 1):
            assert size <= given[0] + (n - 1) * rows * (4 * rank_v + 8) + 512


def test_rows_off_a_16_byte_boundary_are_refused():
    """Operands that the kernels read 16 bytes at a time; U_K only where the
    absorption reads it (not the prepared bases of per-head ones)."""
    from slimkv_amd import _lib
    lib = _lib.lib()
    for name in ('q', 'raw_k', 'lat_v', 'up_k', 'up_v'):
        a = latent_args(1, 32, 700, 256, 256)
        setattr(a, name, (1 << 20) + 8)
        assert lib.slimkv_latent_decode_workspace(ctypes.byref(a)) == 0, name
        assert b'16-byte' in lib.slimkv_last_error()
    a = latent_args(1, 32, 700, 256, 256, per_head=True)
    a.up_k = (1 << 20) + 8
    assert lib.slimkv_latent_decode_workspace(ctypes.byref(a)) == 0
    a.up_k_t = 1 << 20
    assert lib.slimkv_latent_decode_workspace(ctypes.byref(a)) > 0
    a.up_k_bias = (1 << 20) + 2
    assert lib.slimkv_latent_decode_workspace(ctypes.byref(a)) == 0
    for change in ({'q': (1 << 20) + 8}, {'q_sh': 132}):
        r = _lib.ReconDecodeArgs()
        r.base = latent_args(1, 32, 700, 256, 256)
        assert lib.slimkv_recon_decode_workspace(ctypes.byref(r)) > 0
        for name, value in change.items():
            setattr(r.base, name, value)
        assert lib.slimkv_recon_decode_workspace(ctypes.byref(r)) == 0
    r = _lib.ReconDecodeArgs()                  # strides of dimensions of one element do not count
    r.base = latent_args(1, 32, 700, 256, 256)
    r.base.q_sb = r.base.q_sl = 3
    assert lib.slimkv_recon_decode_workspace(ctypes.byref(r)) > 0
