"""GPU: the decode step's own kernel in the formats beside 4-bit keys with 4 query heads a KV head:
3-bit keys (widened to 4 bits in registers, the new row packed across word edges) and 8 query heads
a KV head as two chains over the same rows (the new row stored by both, its range errors counted
once). Against the chunked step, which the formats had before, and oracle/c: outputs, statistics,
lengths and rows, over the score's channel slices, chunk edges, ragged batches, and the look-back
giving up."""

import numpy as np
import pytest

from oracle import native
from oracle.quantize import Format
from oracle.rotate import rotate, signs_from_seed

pytestmark = pytest.mark.gpu

N_KV, D = 2, 64
FORMATS = [(3, 4), (3, 8), (4, 4)]


def _run(ctx, kb, G, lens, steps, q_scale, spin_limit=None, outlier=False):
    import torch
    from insitu_amd import QuantConfig, _lib
    from insitu_amd.cache import CompressedCache
    from insitu_amd.runtime import ptr
    rng = np.random.default_rng(sum(lens) + kb)
    draw = lambda s, *shape: np.rint(rng.standard_normal(shape) * s).astype(np.int64)
    batch = len(lens)
    k, v = (draw(65536, batch, max(lens) + 1, N_KV, D) for _ in "kv")
    caches = []
    for pin in ("step", "chunked"):
        c = CompressedCache(N_KV, D, max(lens) + steps, QuantConfig(key_bits=kb, value_bits=2), batch=batch,
                            n_q_heads=N_KV * G, ctx=ctx)
        for b, n in enumerate(lens):
            if n:
                c.append_rotated(k[b, :n], v[b, :n], seq=b)
        c.pin_kernel(pin)
        if spin_limit is not None and pin == "step":
            _lib.check(ctx.lib.insitu_cache_debug(c.handle, _lib.DEBUG_SPIN_LIMIT, spin_limit))
        caches.append(c)
    f = Format(key_bits=kb)
    for _ in range(steps):
        q, kk, vv = draw(q_scale, batch, N_KV * G, D), draw(65536, batch, N_KV, D), draw(65536, batch, N_KV, D)
        if outlier:
            kk[0, 1, :] = (1 << 31) - 1            # past int32 once rotated: counted, and clamped
        res = []
        for c in caches:
            qd, kd, vd = (ctx.to_device(x, torch.int32) for x in (q, kk, vv))
            out, st = torch.empty((batch, N_KV * G, D), dtype=torch.int32, device=ctx.torch_device), _lib.Stats()
            _lib.check(ctx.lib.insitu_step(c.handle, ptr(qd), ptr(kd), ptr(vd), ptr(out), _lib.SEQUENTIAL, st))
            res.append((out.cpu().numpy(), {n: getattr(st, n) for n, _ in st._fields_}))
        np.testing.assert_array_equal(res[0][0], res[1][0])
        if spin_limit is None:
            assert res[0][1] == res[1][1]
    for b, n in enumerate(lens):
        for h in range(N_KV):
            np.testing.assert_array_equal(*(c.read_rows(h, 0, n + steps, seq=b) for c in caches))
    assert caches[0].lengths() == [n + steps for n in lens]
    qr = rotate(q[0], signs_from_seed(D, 0, 1))
    if lens[0] == max(lens) and not outlier:
        want = np.concatenate([native.attend_online(qr[G * h:G * h + G], caches[0].view(h), f)[0] for h in range(N_KV)])
        np.testing.assert_array_equal(res[0][0][0], want)
    return res[0][1]


@pytest.mark.parametrize("n", [0, 1, 62, 63, 64, 127, 130, 300, 600, 1022, 1023, 1024, 2047, 2500])
@pytest.mark.parametrize("kb,G", FORMATS)
@pytest.mark.parametrize("q_scale", [1 << 13, 1 << 17])
def test_contexts(ctx, kb, G, n, q_scale):
    assert _run(ctx, kb, G, [n], 2, q_scale)["serial_fallbacks"] == 0


@pytest.mark.parametrize("kb,G", FORMATS)
def test_ragged_batch(ctx, kb, G):
    _run(ctx, kb, G, [2100, 0, 65, 1023], 2, 1 << 15)


@pytest.mark.parametrize("kb,G", FORMATS)
def test_the_look_back_giving_up(ctx, kb, G):
    """Spin limit 0: every head with a chunk before it takes the reference loop."""
    assert _run(ctx, kb, G, [1500], 1, 1 << 15, spin_limit=0)["serial_fallbacks"] > 0


@pytest.mark.parametrize("kb,G", FORMATS)
def test_range_errors_are_counted_once(ctx, kb, G):
    assert _run(ctx, kb, G, [70], 1, 1 << 13, outlier=True)["range_errors"] > 0


@pytest.mark.parametrize("chunk_tokens", [512, 1024])
@pytest.mark.parametrize("longer", [0, 1])
def test_either_side_of_the_choice(ctx, longer, chunk_tokens):
    """8 query heads a KV head: 256 chunks in all (64 sequences, 4 chains) and 260, where caches of
    1,024-token chunks go back to the chunked step; the automatic choice against both kernels."""
    import torch
    from insitu_amd import QuantConfig, _lib
    from insitu_amd.cache import CompressedCache
    from insitu_amd.runtime import ptr
    batch, n, G = 64, 1023, 8
    rng = np.random.default_rng(longer)
    draw = lambda s, *shape: ctx.to_device(np.rint(rng.standard_normal(shape) * s).astype(np.int64), torch.int32)
    k, v = draw(65536, n + 1, N_KV, D), draw(65536, n + 1, N_KV, D)
    q, kk, vv = draw(16384, batch, N_KV * G, D), draw(65536, batch, N_KV, D), draw(65536, batch, N_KV, D)
    res = []
    for pin in ("auto", "step", "chunked"):
        c = CompressedCache(N_KV, D, n + 3, QuantConfig(key_bits=3, value_bits=2), batch=batch, n_q_heads=N_KV * G,
                            chunk_tokens=chunk_tokens, ctx=ctx)
        for b in range(batch):
            m = n + (longer if b == 5 else 0)
            c.append_rotated(k[:m], v[:m], seq=b)
        c.pin_kernel(pin)
        out, st = torch.empty_like(q), _lib.Stats()
        _lib.check(ctx.lib.insitu_step(c.handle, ptr(q), ptr(kk), ptr(vv), ptr(out), _lib.SEQUENTIAL, st))
        res.append((out, [getattr(st, f) for f, _ in st._fields_], [c.read_rows(1, n, 1, seq=b) for b in (0, 5, 63)]))
        assert c.lengths() == [n + 1 + (longer if b == 5 else 0) for b in range(batch)]
    for r in res[1:]:
        assert torch.equal(r[0], res[0][0]) and r[1] == res[0][1]
        np.testing.assert_array_equal(r[2], res[0][2])
