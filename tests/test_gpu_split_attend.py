"""GPU: the two-launch attend of two-pass mode (attend_split.hip) at the sizes and values where it
can go wrong: contexts around its 16-token tiles, 64-token blocks and workgroups, every query-head
group, key and value width it takes, ragged batches with empty sequences, the decode step (the new
row at every place of a tile and a block), scores that need int64, value terms past three digits,
sums that clamp, scores that may not be exact (the reference loop), and queries past the rotated
range. Every output, statistic and row against oracle/c, and the automatic choice against the
chunked attend."""

import numpy as np
import pytest

from oracle import native
from oracle.quantize import Cache, Format

pytestmark = pytest.mark.gpu

N_KV = 2
FORMATS = [(64, 4, 2, 4), (64, 3, 2, 8), (64, 2, 3, 1), (64, 4, 1, 5), (64, 2, 2, 4), (128, 3, 3, 4), (128, 4, 2, 2),
           (128, 2, 1, 8)]


def _draw(rng, scale, *shape):
    return np.rint(rng.standard_normal(shape) * scale).astype(np.int64)


def _check(out, st, q, hosts, f, G, serial=0):
    """out (batch, heads, d) against the oracle over each sequence's rows (None: no rows)."""
    sts = []
    for b, host in enumerate(hosts):
        for h in range(N_KV):
            got = out[b, G * h:G * h + G]
            if host is None:
                assert not got.any()
                continue
            want, s = native.attend_two_pass(q[b, G * h:G * h + G], host.view(h), f)
            np.testing.assert_array_equal(got, want, err_msg=f"sequence {b} head {h}")
            sts.append(s)
    assert st.max_abs_score == max(s.max_abs_score for s in sts)
    assert st.score_overflows == sum(s.score_overflows for s in sts)
    assert st.max_abs_acc == max(s.max_abs_acc for s in sts)
    assert st.acc_overflows == sum(s.acc_overflows for s in sts)
    if serial is not None:
        assert st.serial_fallbacks == serial


def _attend(ctx, fmt, lens, q, k, v, serial=0, pin="split"):
    """Sequence b attends its first lens[b] rows of k, v (batch, rows, N_KV, d)."""
    from insitu_amd import QuantConfig
    from insitu_amd.attention import CompressedAttention
    from insitu_amd.cache import CompressedCache
    d, kb, vb, G = fmt
    f = Format(d=d, key_bits=kb, value_bits=vb)
    c = CompressedCache(N_KV, d, max(lens) + 3, QuantConfig(key_bits=kb, value_bits=vb), batch=len(lens),
                        n_q_heads=N_KV * G, ctx=ctx)
    hosts = []
    for b, n in enumerate(lens):
        host = None
        if n:
            c.append_rotated(k[b, :n], v[b, :n], seq=b)
            host = Cache(N_KV, n, f)
            host.append_rotated(k[b, :n], v[b, :n])
        hosts.append(host)
    c.pin_kernel(pin)
    out, st = CompressedAttention(c).attend(q, "two_pass")
    _check(out.cpu().numpy(), st, q, hosts, f, G, serial)
    assert st.n_tokens == max(lens)
    return st


@pytest.mark.parametrize("lens", [(1,), (15, 16, 17), (63, 64, 65, 0), (255, 257, 1, 0, 256), (1025,), (4200, 3)])
@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("q_scale", [1 << 13, 1 << 17])
def test_contexts_and_formats(ctx, fmt, lens, q_scale):
    """A flat softmax (the queries scaled by 1/sqrt(d)) and a peaked one, where blocks are skipped."""
    d, _, _, G = fmt
    rng = np.random.default_rng(sum(lens))
    q = _draw(rng, q_scale, len(lens), N_KV * G, d)
    k, v = (_draw(rng, 65536, len(lens), max(lens), N_KV, d) for _ in "kv")
    _attend(ctx, fmt, lens, q, k, v)


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("q_scale,kv_scale", [(1 << 21, 1 << 21), (1 << 24, 1 << 18), (1 << 25, 1 << 22)])
def test_large_values(ctx, fmt, q_scale, kv_scale):
    """Scores past 32 bits; queries that need their fourth digit; both, with norms at their 16-bit limit."""
    d, _, _, G = fmt
    rng = np.random.default_rng(7)
    q = _draw(rng, q_scale, 1, N_KV * G, d)
    k, v = (_draw(rng, kv_scale, 1, 61, N_KV, d) for _ in "kv")
    _attend(ctx, fmt, (61,), q, k, v, serial=0 if kv_scale < 1 << 22 else None)


@pytest.mark.parametrize("fmt", [(64, 4, 2, 4), (64, 3, 2, 8), (128, 3, 3, 4)])
def test_sums_that_clamp(ctx, fmt):
    """Equal large values under a flat softmax: terms past three digits, and sums past the clamp
    (a token adds at least 3,169,055: 678 of them), which are added up exactly before it."""
    d, _, _, G = fmt
    q = np.zeros((1, N_KV * G, d), dtype=np.int64)
    k = np.full((1, 900, N_KV, d), 4000, dtype=np.int64)
    v = np.full((1, 900, N_KV, d), (1 << 22) - 7, dtype=np.int64)
    assert _attend(ctx, fmt, (900,), q, k, v).acc_overflows > 0
    assert _attend(ctx, fmt, (300,), q, k, v).acc_overflows == 0


@pytest.mark.parametrize("d,kb,vb", [(64, 4, 2), (64, 3, 3), (128, 3, 3), (128, 4, 2)])
@pytest.mark.parametrize("c_max,taken", [(982_782, True), (982_783, False), ((1 << 20) - 1, False)])
def test_value_centroids_up_to_20_bits(ctx, monkeypatch, d, kb, vb, c_max, taken):
    """Terms up to the digits' limit with the largest norm and p = 1; a codebook past it is refused by
    the split attend, and the automatic choice gives the oracle's outputs all the same."""
    import dataclasses

    from insitu_amd import QuantConfig, _lib
    from insitu_amd.attention import CompressedAttention
    from insitu_amd.cache import Codebook, CompressedCache
    n = 1 << vb
    vc = np.rint(np.linspace(-1, 1, n) * c_max).astype(np.int64)

    class Wide(Format):
        def codebooks(self):
            k_c, k_b, _, v_b = super().codebooks()
            return k_c, k_b, vc, v_b

    build = Codebook.build
    books = iter([None, vc])                          # CompressedCache builds the key's first
    monkeypatch.setattr(Codebook, "build", staticmethod(
        lambda *a: build(*a) if (v := next(books)) is None else dataclasses.replace(build(*a), centroids=v)))
    T, G = 70, 4
    c = CompressedCache(N_KV, d, T, QuantConfig(key_bits=kb, value_bits=vb), n_q_heads=N_KV * G, ctx=ctx)
    rng = np.random.default_rng(d + vb)
    # the largest norm; a quarter of the channels at twice it, in the outermost codes
    v = np.where(rng.random((T, N_KV, d)) < 0.25, 1 << 24, 0) * rng.choice([-1, 1], (T, N_KV, d))
    k = _draw(rng, 65536, T, N_KV, d)
    q = _draw(rng, 8192, 1, N_KV * G, d)
    q[0, 1:3] = 0                                     # p = 1 throughout
    f = Wide(d=d, key_bits=kb, value_bits=vb)
    host = Cache(N_KV, T, f)
    host.append_rotated(k, v)
    assert host.view(0).v_norm.max() == 32767 and {0, n - 1} <= set(host.view(0).v_idx.ravel().tolist())
    c.append_rotated(k, v)
    a = CompressedAttention(c)
    for pin in ("auto", "split") if taken else ("auto",):
        c.pin_kernel(pin)
        out, st = a.attend(q, "two_pass")
        _check(out.cpu().numpy(), st, q, [host], f, G, serial=None)
    if not taken:
        with pytest.raises(_lib.FormatError, match="EINVAL"):
            c.pin_kernel("split")


def test_range_errors_and_scores_that_may_not_be_exact(ctx):
    """Queries past the rotated range are counted; a head with a value of 2^30 takes the reference
    loop, alone."""
    fmt = (64, 4, 2, 4)
    rng = np.random.default_rng(3)
    q = _draw(rng, 8192, 1, N_KV * 4, 64)
    k, v = (_draw(rng, 65536, 1, 130, N_KV, 64) for _ in "kv")
    q[0, 1, 7] = 1 << 30
    q[0, 6, 5] = -(1 << 27)
    assert _attend(ctx, fmt, (130,), q, k, v, serial=1).range_errors == 2


@pytest.mark.parametrize("fmt", [(64, 4, 2, 4), (64, 3, 2, 8), (128, 3, 3, 4), (128, 4, 2, 3)])
@pytest.mark.parametrize("base", [0, 14, 62, 254])
def test_steps(ctx, fmt, base):
    """Decode steps over the edges of a tile, a block and a workgroup, two ragged sequences: outputs,
    statistics, lengths and rows as the chunked step gives them."""
    import torch

    from insitu_amd import QuantConfig, _lib
    from insitu_amd.cache import CompressedCache
    from insitu_amd.runtime import ptr
    d, kb, vb, G = fmt
    rng = np.random.default_rng(base)
    k, v = (_draw(rng, 65536, 2, base + 2, N_KV, d) for _ in "kv")
    caches = []
    for pin in ("split", "chunked"):
        c = CompressedCache(N_KV, d, base + 8, QuantConfig(key_bits=kb, value_bits=vb), batch=2, n_q_heads=N_KV * G, ctx=ctx)
        for b, n in enumerate((base, base // 2)):
            if n:
                c.append_rotated(k[b, :n], v[b, :n], seq=b)
        c.pin_kernel(pin)
        caches.append(c)
    for _ in range(4):
        q, kk, vv = (ctx.to_device(_draw(rng, s, 2, h, d), torch.int32)
                     for s, h in ((8192, N_KV * G), (65536, N_KV), (65536, N_KV)))
        res = []
        for c in caches:
            out, st = torch.empty((2, N_KV * G, d), dtype=torch.int32, device=ctx.torch_device), _lib.Stats()
            _lib.check(ctx.lib.insitu_step(c.handle, ptr(q), ptr(kk), ptr(vv), ptr(out), _lib.TWO_PASS, st))
            res.append((out.cpu().numpy(), [getattr(st, n) for n, _ in st._fields_]))
        np.testing.assert_array_equal(res[0][0], res[1][0])
        assert res[0][1] == res[1][1]
    for b, n in enumerate((base + 4, base // 2 + 4)):
        assert [c.lengths()[b] for c in caches] == [n, n]
        for h in range(N_KV):
            np.testing.assert_array_equal(*(c.read_rows(h, 0, n, seq=b) for c in caches))


@pytest.mark.parametrize("fmt,n", [((64, 4, 2, 4), 300), ((128, 3, 3, 4), 300), ((128, 3, 3, 4), 17000)])
def test_auto_choice_equals_the_chunked_attend(ctx, fmt, n):
    """Either side of the rule."""
    from insitu_amd import QuantConfig
    from insitu_amd.attention import CompressedAttention
    from insitu_amd.cache import CompressedCache
    d, kb, vb, G = fmt
    rng = np.random.default_rng(n)
    c = CompressedCache(N_KV, d, n, QuantConfig(key_bits=kb, value_bits=vb), n_q_heads=N_KV * G, ctx=ctx)
    c.append_rotated(*(_draw(rng, 65536, n, N_KV, d) for _ in "kv"))
    q = _draw(rng, 16384, 1, N_KV * G, d)
    outs = []
    for pin in ("auto", "split", "chunked"):
        c.pin_kernel(pin)
        out, st = CompressedAttention(c).attend(q, "two_pass")
        outs.append((out.cpu().numpy(), st))
    for o, st in outs[1:]:
        np.testing.assert_array_equal(o, outs[0][0])
        assert st == outs[0][1]


def test_formats_it_does_not_take_are_refused(ctx):
    from insitu_amd import QuantConfig, _lib
    from insitu_amd.cache import CompressedCache
    c = CompressedCache(N_KV, 64, 32, QuantConfig(key_bits=5, value_bits=3), n_q_heads=8, ctx=ctx)
    with pytest.raises(_lib.FormatError, match="EINVAL"):
        c.pin_kernel("split")
