"""GPU: the prefill attend on matrix cores (attend_prefill.hip) at the sizes and values where it
can go wrong: contexts and query counts around its 16-token tiles, its stages and its 16-row
waves, every query-head group, key and value width it takes, scores that need int64 (a fourth
digit of q, products past 32 bits), value terms past three digits, an accumulator that clamps
(rows recomputed by the reference loop), and values past the rotated query's range. Every output
and statistic against oracle/c over the same rows."""

import numpy as np
import pytest

from oracle import native
from oracle.quantize import Cache, Format

pytestmark = pytest.mark.gpu

N_KV = 2
FORMATS = [(64, 4, 2, 4), (64, 3, 2, 8), (64, 2, 3, 1), (64, 4, 1, 3), (128, 3, 3, 4), (128, 4, 2, 2)]


def _cache(ctx, capacity, d, kb, vb, G, pin=2):
    from insitu_amd import QuantConfig, _lib
    from insitu_amd.cache import CompressedCache
    c = CompressedCache(N_KV, d, capacity, QuantConfig(key_bits=kb, value_bits=vb), n_q_heads=N_KV * G, ctx=ctx)
    _lib.check(ctx.lib.insitu_cache_debug(c.handle, _lib.DEBUG_PREFILL, pin))
    return c


def _run(ctx, fmt, base, n, q, k, v, mode, serial=0):
    from insitu_amd.attention import CompressedAttention
    d, kb, vb, G = fmt
    f = Format(d=d, key_bits=kb, value_bits=vb)
    c = _cache(ctx, base + n + 5, *fmt)
    c.append_rotated(k, v)
    out, st = CompressedAttention(c).attend_prefill(q, base, mode)
    out = out.cpu().numpy()
    host = Cache(N_KV, base + n, f)
    host.append_rotated(k, v)
    fn = native.attend_online if mode == "online" else native.attend_two_pass
    sts, views = [], [host.view(h) for h in range(N_KV)]
    for i in range(n):
        for h in range(N_KV):
            want, s = fn(q[i, G * h:G * h + G], views[h].select(slice(0, base + i + 1)), f)
            np.testing.assert_array_equal(out[i, G * h:G * h + G], want, err_msg=f"query {i} head {h}")
            sts.append(s)
    assert st.n_tokens == base + n
    if mode == "online":
        assert st.rescale_events == sum(s.rescale_events for s in sts)
    assert st.max_abs_score == max(s.max_abs_score for s in sts)
    assert st.score_overflows == sum(s.score_overflows for s in sts)
    assert st.max_abs_acc == max(s.max_abs_acc for s in sts)
    assert st.acc_overflows == sum(s.acc_overflows for s in sts)
    if serial is not None:
        assert st.serial_fallbacks == serial
    return st


def _inputs(seed, fmt, base, n, q_scale, kv_scale):
    d, _, _, G = fmt
    rng = np.random.default_rng(seed)
    draw = lambda rows, heads, s: np.rint(rng.standard_normal((rows, heads, d)) * s).astype(np.int64)
    return draw(n, N_KV * G, q_scale), draw(base + n, N_KV, kv_scale), draw(base + n, N_KV, kv_scale)


@pytest.mark.parametrize("mode", ["online", "two_pass"])
@pytest.mark.parametrize("base,n", [(0, 1), (0, 16), (0, 17), (15, 33), (63, 65), (200, 7)])
@pytest.mark.parametrize("fmt", FORMATS)
def test_tiles_and_formats(ctx, fmt, base, n, mode):
    """Unit values, the queries scaled by 1/sqrt(d): a flat softmax."""
    q, k, v = _inputs(base + n, fmt, base, n, 65536 / 8, 65536)
    _run(ctx, fmt, base, n, q, k, v, mode)


@pytest.mark.parametrize("mode", ["online", "two_pass"])
@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("q_scale,kv_scale", [(1 << 16, 1 << 16), (1 << 21, 1 << 21), (1 << 24, 1 << 18), (1 << 25, 1 << 22)])
def test_large_values(ctx, fmt, mode, q_scale, kv_scale):
    """Peaked scores; scores past 32 bits; queries that need their fourth digit; both, with norms
    at their 16-bit limit."""
    base, n = 21, 40
    q, k, v = _inputs(7, fmt, base, n, q_scale, kv_scale)
    _run(ctx, fmt, base, n, q, k, v, mode, serial=0 if kv_scale < 1 << 22 else None)


@pytest.mark.parametrize("mode", ["online", "two_pass"])
@pytest.mark.parametrize("target", [-(1 << 31), -(1 << 31) + 1])
def test_scores_at_the_end_of_32_bits(ctx, mode, target):
    """A first score of -2^31, the narrow scores' mark of a row with no token yet, is an event too."""
    fmt = (64, 4, 2, 4)
    d, kb, vb, G = fmt
    f = Format(d=d, key_bits=kb, value_bits=vb)
    q, k, v = _inputs(4, fmt, 0, 3, 64, 1 << 21)
    host = Cache(N_KV, 3, f)
    host.append_rotated(k, v)
    kv, kc = host.view(0), f.codebooks()[0]
    c, kn = kc[kv.k_idx[0].astype(int)], int(kv.k_norm[0])
    # dot in [target 2^24 / kn, (target + 1) 2^24 / kn): all channels alike, then two channels' steps
    lo, hi = -((-target << 24) // kn), -((-(target + 1) << 24) // kn)
    x = (np.sign(c) * (lo // int(np.abs(c).sum()))).astype(np.int64)
    i, j = np.argmax(c), np.argmin(np.abs(np.abs(c) - 4200))
    rest = lo - int(x @ c)
    for s in range(-20000, 20000):
        t = (rest - s * int(c[j])) // int(c[i]) + 1
        if lo <= int(x @ c) + s * int(c[j]) + t * int(c[i]) < hi:
            break
    x[j] += s
    x[i] += t
    assert (int(x @ c) * kn) >> 24 == target and np.abs(x).max() < 0x7F7F7F and i != j
    q[0, 1] = x
    _run(ctx, fmt, 0, 3, q, k, v, mode)


@pytest.mark.parametrize("fmt,waves", [((64, 4, 2, 4), 4), ((128, 3, 3, 4), 8)])
@pytest.mark.parametrize("mode", ["online", "two_pass"])
@pytest.mark.parametrize("q_wide,q_scale,kv_scale", [(1 << 24, 8192, 65536), (1 << 21, 1 << 10, 1 << 21)])
def test_one_wave_sends_its_workgroup_to_int64_scores(ctx, fmt, waves, mode, q_wide, q_scale, kv_scale):
    """One row of a workgroup needs int64 scores (its fourth digit; products past 32 bits), another
    wave's in each workgroup and none's in every ninth: all its waves start again together."""
    per_wave = 16 // fmt[3]                            # queries
    n = 40 * waves * per_wave
    q, k, v = _inputs(11, fmt, 0, n, q_scale, kv_scale)
    v = v * 65536 // kv_scale                          # no accumulator near its clamp
    for b in range(40):
        if b % 9 != 8:
            row = q[(b * waves + b % waves) * per_wave + b % per_wave, b % (N_KV * fmt[3])]
            row[:] = q_wide
            row[::3] = -q_wide
    _run(ctx, fmt, 0, n, q, k, v, mode)


@pytest.mark.parametrize("fmt", [(64, 4, 2, 4), (128, 3, 3, 4)])
@pytest.mark.parametrize("mode", ["online", "two_pass"])
def test_clamped_accumulators_and_wide_terms(ctx, fmt, mode):
    """Equal large values under a flat softmax: terms past three digits (the largest norm), and
    accumulators that reach the clamp, in the rows with the longest contexts only."""
    d, _, _, G = fmt
    # a token adds at most 2^22 (the value) and, in the coarser 3-bit code, 3,169,055: 678 of them clamp
    base, n = 700, 20
    q = np.zeros((n, N_KV * G, d), dtype=np.int64)
    k = np.full((base + n, N_KV, d), 4000, dtype=np.int64)
    v = np.full((base + n, N_KV, d), (1 << 22) - 7, dtype=np.int64)
    st = _run(ctx, fmt, base, n, q, k, v, mode, serial=None)
    assert st.acc_overflows > 0 and st.serial_fallbacks > 0
    _run(ctx, fmt, 300, n, q, k[:300 + n], v[:300 + n], mode, serial=0)


@pytest.mark.parametrize("fmt", [(64, 4, 2, 4), (64, 2, 3, 1), (128, 3, 3, 2), (128, 4, 2, 8)])
@pytest.mark.parametrize("mode", ["online", "two_pass"])
def test_value_centroids_at_20_bits(ctx, monkeypatch, fmt, mode):
    """The largest terms: centroids of 2^20 - 1, the largest norm, p = 1. The first 16 rows' sums fit the
    accumulator's bound, the later rows take the reference loop."""
    import dataclasses

    from insitu_amd.attention import CompressedAttention
    from insitu_amd.cache import Codebook
    d, kb, vb, G = fmt
    vc = np.rint(np.linspace(-1, 1, 1 << vb) * ((1 << 20) - 1)).astype(np.int64)

    class Wide(Format):
        def codebooks(self):
            k_c, k_b, _, v_b = super().codebooks()
            return k_c, k_b, vc, v_b

    build = Codebook.build
    books = iter([None, vc])                          # CompressedCache builds the key's first
    monkeypatch.setattr(Codebook, "build", staticmethod(
        lambda *a: build(*a) if (v := next(books)) is None else dataclasses.replace(build(*a), centroids=v)))
    n = 24
    c = _cache(ctx, n, *fmt)
    q, k, v = _inputs(2, fmt, 0, n, 4096, 65536)
    q[:, ::2] = 0
    rng = np.random.default_rng(1)
    v = np.where(rng.random(v.shape) < 0.25, 1 << 24, 0) * rng.choice([-1, 1], v.shape)
    f = Wide(d=d, key_bits=kb, value_bits=vb)
    host = Cache(N_KV, n, f)
    host.append_rotated(k, v)
    assert host.view(0).v_norm.max() == 32767 and {0, (1 << vb) - 1} <= set(host.view(0).v_idx.ravel().tolist())
    c.append_rotated(k, v)
    out, st = CompressedAttention(c).attend_prefill(q, 0, mode)
    out = out.cpu().numpy()
    fn = native.attend_online if mode == "online" else native.attend_two_pass
    for i in range(n):
        for h in range(N_KV):
            want, _ = fn(q[i, G * h:G * h + G], host.view(h).select(slice(0, i + 1)), f)
            np.testing.assert_array_equal(out[i, G * h:G * h + G], want, err_msg=f"query {i} head {h}")
    assert st.serial_fallbacks < n * N_KV * G


@pytest.mark.parametrize("fmt", [(64, 4, 2, 4), (64, 2, 3, 1), (128, 3, 3, 2)])
@pytest.mark.parametrize("mode", ["online", "two_pass"])
def test_denominators_past_32_bits_a_lane(ctx, fmt, mode):
    """Equal and nearly equal scores over more than 2^19 rows: a lane's share of the denominator, four
    rows of 16 at 2^15 each, passes 2^32."""
    from insitu_amd.attention import CompressedAttention
    d, kb, vb, G = fmt
    f = Format(d=d, key_bits=kb, value_bits=vb)
    T, n, tile = (1 << 19) + 700, 3, 4096
    q, k, v = _inputs(5, fmt, tile - n, n, 16, 8192)
    q[0] = 0
    c, host = _cache(ctx, T, *fmt), Cache(N_KV, tile, f)
    host.append_rotated(k, v)
    for t in range(0, T, tile):
        c.append_rotated(k[:T - t], v[:T - t])
    out, st = CompressedAttention(c).attend_prefill(q, T - n, mode)
    out = out.cpu().numpy()
    fn = native.attend_online if mode == "online" else native.attend_two_pass
    for h in range(N_KV):
        kv = host.view(h)
        rep = lambda a: np.concatenate([a] * (T // tile + 1))
        kv = type(kv)(rep(kv.k_idx), rep(kv.k_norm), rep(kv.v_idx), rep(kv.v_norm))
        for i in range(n):
            want, _ = fn(q[i, G * h:G * h + G], kv.select(slice(0, T - n + i + 1)), f)
            np.testing.assert_array_equal(out[i, G * h:G * h + G], want, err_msg=f"query {i} head {h}")
    assert st.serial_fallbacks == 0 and st.n_tokens == T


def test_range_errors_and_rows_past_exact_scores(ctx):
    """Queries past the rotated range are counted; a row whose scores may not be exact (a value
    of 2^30) takes the reference loop, alone."""
    fmt, base, n = (64, 4, 2, 4), 30, 9
    q, k, v = _inputs(3, fmt, base, n, 8192, 65536)
    q[4, 1, 7] = 1 << 30
    q[2, 3, 5] = -(1 << 27)
    st = _run(ctx, fmt, base, n, q, k, v, "online", serial=1)
    assert st.range_errors == 2


@pytest.mark.parametrize("fmt", [(64, 4, 2, 4), (128, 3, 3, 4)])
def test_rows_at_4_byte_aligned_addresses(ctx, fmt):
    """q and out as views one int32 into a larger tensor."""
    import torch

    from insitu_amd.attention import CompressedAttention
    d, _, _, G = fmt
    n = 21
    q, k, v = _inputs(8, fmt, 0, n, 8192, 65536)
    c = _cache(ctx, n, *fmt)
    c.append_rotated(k, v)
    a = CompressedAttention(c)
    want = a.attend_prefill(q, 0, "online")[0]
    bufs = [torch.zeros(q.size + 1, dtype=torch.int32, device=ctx.torch_device) for _ in "qo"]
    q1, o1 = (b[1:].view(q.shape) for b in bufs)
    q1.copy_(torch.from_numpy(q))
    assert q1.data_ptr() % 16 == o1.data_ptr() % 16 == 4
    got = a.attend_prefill(q1, 0, "online", out=o1)[0]
    assert torch.equal(got, want) and int(bufs[1][0]) == 0


@pytest.mark.parametrize("mode", ["online", "two_pass"])
def test_auto_choice_equals_both_kernels(ctx, mode):
    """The automatic choice and either pinned kernel give the same output, either side of the rule."""
    from insitu_amd import _lib
    from insitu_amd.attention import CompressedAttention
    fmt = (64, 4, 2, 4)
    for base, n in ((900, 3), (40, 200)):
        q, k, v = _inputs(n, fmt, base, n, 8192, 65536)
        c = _cache(ctx, base + n, *fmt, pin=0)
        c.append_rotated(k, v)
        outs = []
        for pin in (0, 1, 2):
            _lib.check(ctx.lib.insitu_cache_debug(c.handle, _lib.DEBUG_PREFILL, pin))
            outs.append(CompressedAttention(c).attend_prefill(q, base, mode)[0].cpu().numpy())
        np.testing.assert_array_equal(outs[0], outs[1])
        np.testing.assert_array_equal(outs[0], outs[2])


def test_formats_it_does_not_take_are_refused(ctx):
    from insitu_amd import _lib
    with pytest.raises(_lib.FormatError, match="EINVAL"):
        _cache(ctx, 32, 64, 5, 3, 4)
