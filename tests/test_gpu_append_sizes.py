"""GPU: the append's two kernels by size (write_path.hip): the lane-per-channel kernel, a row a wave
up to 8,192 rows and several beyond, and the lane = row kernel's partial tiles, one against the other
and the automatic choice against both, over sizes around a workgroup, a tile, the line between the
kernels (4,096 rows) and the grid's limit (8,192); three sequences at once and one of them, wire rows;
and the rows against the oracle's encoder."""

import numpy as np
import pytest

from oracle.quantize import Cache, Format
from oracle.rotate import rotate, signs_from_seed

pytestmark = pytest.mark.gpu

N_KV = 4


@pytest.mark.parametrize("n", [1, 3, 8, 15, 17, 64, 341, 342, 513, 682, 683, 1024, 1025, 2049])   # 12 n rows
@pytest.mark.parametrize("d,kb,vb", [(64, 4, 2), (64, 2, 2), (64, 3, 2), (128, 3, 3)])
def test_append_kernels_by_size(ctx, d, kb, vb, n):
    from insitu_amd import QuantConfig, _lib
    from insitu_amd.cache import CompressedCache
    rng = np.random.default_rng(n)
    k, v = (rng.integers(-(1 << 20), 1 << 20, size=(3, n, N_KV, d)) for _ in "kv")
    f = Format(d=d, key_bits=kb, value_bits=vb)
    caches = []
    for pin in (0, 1, 2):
        c = CompressedCache(N_KV, d, n + 2, QuantConfig(key_bits=kb, value_bits=vb), batch=3, n_q_heads=4 * N_KV, ctx=ctx)
        _lib.check(ctx.lib.insitu_cache_debug(c.handle, _lib.DEBUG_APPEND, pin))
        c.append_wire(k, v)
        c.append_wire(k[1, :1], v[1, :1], seq=1)
        assert c.lengths() == [n, n + 1, n]
        caches.append(c)
    sg = signs_from_seed(d, 0, 1)
    for b in range(3):
        for h in range(N_KV):
            rows = [c.read_rows(h, 0, n + (b == 1), seq=b) for c in caches]
            np.testing.assert_array_equal(rows[1], rows[0])
            np.testing.assert_array_equal(rows[2], rows[0])
    host = Cache(N_KV, n, f)
    host.append_rotated(*(rotate(x[2].reshape(-1, d), sg).reshape(n, N_KV, d) for x in (k, v)))
    for h in (0, N_KV - 1):
        np.testing.assert_array_equal(caches[0].read_rows(h, 0, n, seq=2), host.buf[:n, h])


@pytest.mark.parametrize("n", [4095, 4096, 4097, 8191, 8192, 8193])
@pytest.mark.parametrize("kb,vb", [(4, 2), (2, 2), (3, 2)])
def test_rows_at_the_lines(ctx, kb, vb, n):
    """One KV head of one sequence: n rows exactly."""
    from insitu_amd import QuantConfig, _lib
    from insitu_amd.cache import CompressedCache
    rng = np.random.default_rng(n)
    k, v = (rng.integers(-(1 << 20), 1 << 20, size=(n, 1, 64)) for _ in "kv")
    host = Cache(1, n, Format(key_bits=kb, value_bits=vb))
    sg = signs_from_seed(64, 0, 1)
    host.append_rotated(*(rotate(x.reshape(-1, 64), sg).reshape(x.shape) for x in (k, v)))
    for pin in (0, 1, 2):
        c = CompressedCache(1, 64, n, QuantConfig(key_bits=kb, value_bits=vb), n_q_heads=4, ctx=ctx)
        _lib.check(ctx.lib.insitu_cache_debug(c.handle, _lib.DEBUG_APPEND, pin))
        c.append_wire(k, v)
        np.testing.assert_array_equal(c.read_rows(0, 0, n), host.buf[:, 0], err_msg=f"kernel {pin}")
