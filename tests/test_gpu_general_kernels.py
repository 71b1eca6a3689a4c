"""GPU: the kernels that the automatic choice reaches only outside other tests' sizes, pinned.

Two-pass attends and steps run on the split attend, prompts on the prefill kernel and 3-bit decode
steps on the step kernel wherever they are the faster ones; the chunked attend, the virtual batch of
causal attends and the two-launch step remain for the rest (long or mid-size contexts, few queries
behind a long context, other formats). The tests whose sizes the choice moved to the newer kernels
run again here with every cache pinned to the general ones, on both chunk sizes where it matters;
tests of the same names run unpinned in their own files."""

import functools

import numpy as np
import pytest

import test_gpu_formats as F
import test_gpu_parity as P
import test_gpu_scratch as S
import test_zz_no_alloc as Z
from oracle import native
from oracle.quantize import Cache, Format

pytestmark = pytest.mark.gpu


def _pin_every_cache(monkeypatch, chunked):
    from insitu_amd import _lib
    from insitu_amd.cache import CompressedCache
    init = CompressedCache.__init__

    def pinned(self, *a, **kw):
        init(self, *a, **kw)
        _lib.check(self.ctx.lib.insitu_cache_debug(self.handle, _lib.DEBUG_PREFILL, _lib.PREFILL_BATCH))
        if chunked:
            self.pin_kernel("chunked")         # raises unless the chunked attend takes the cache

    monkeypatch.setattr(CompressedCache, "__init__", pinned)


@pytest.fixture
def virtual_batch(monkeypatch):
    _pin_every_cache(monkeypatch, False)


@pytest.fixture
def chunked(monkeypatch):
    _pin_every_cache(monkeypatch, True)


@pytest.fixture(params=[512, 1024])
def chunk_tokens(request, monkeypatch):
    for m in (P, Z):
        monkeypatch.setattr(m, "_cache", functools.partial(m._cache, chunk_tokens=request.param))
    return request.param


# -- two-pass attends and steps on the chunked attend --------------------------------

@pytest.mark.parametrize("T", [1, 63, 65, 511, 512, 513, 700, 1025, 3000])
def test_two_pass_contexts(ctx, chunked, chunk_tokens, T):
    P.test_attend_random_contexts_against_native_oracle(ctx, "two_pass", T)


def test_two_pass_full_context(ctx, chunked, chunk_tokens):
    P.test_full_c2_context_against_native_oracle(ctx, "two_pass")


def test_two_pass_many_chains(ctx, chunked, chunk_tokens):
    P.test_many_chains_merge_their_statistics(ctx, "two_pass")


def test_ragged_batch(ctx, chunked, chunk_tokens):
    P.test_ragged_batch_multi_chunk(ctx)


def test_later_chunk_replay(ctx, chunked, chunk_tokens):
    P.test_a_later_chunk_replays_from_chunk_zeros_published_state(ctx)


def test_acc_clamp(ctx, chunked, chunk_tokens):
    P.test_acc_clamp_path_is_exact(ctx)


@pytest.mark.parametrize("n_kv,lens", [(2, [5000, 3100, 4097]), (1, [9000, 2500, 1, 7000, 4200]), (3, [20000])])
def test_chains_that_straddle_xcds(ctx, chunked, chunk_tokens, n_kv, lens):
    P.test_chains_that_straddle_xcds(ctx, n_kv, lens)


def test_d128_3b3b(ctx, chunked, chunk_tokens):
    P.test_d128_3b3b_against_native_oracle(ctx)


@pytest.mark.parametrize("G", [1, 2])
@pytest.mark.parametrize("T", [1, 700, 9000])
def test_fewer_than_four_query_heads(ctx, chunked, monkeypatch, G, T):
    from insitu_amd.cache import CompressedCache
    pin = CompressedCache.pin_kernel
    monkeypatch.setattr(CompressedCache, "pin_kernel", lambda self, path: pin(self, "chunked"))
    F.test_fewer_than_four_query_heads(ctx, G, T)


@pytest.mark.parametrize("d,kb,vb", [(64, 4, 2), (128, 3, 3)])
def test_two_pass_steps_in_three_launches(ctx, chunked, d, kb, vb):
    """The write kernel, the maxima and the sums."""
    P.test_fused_step_ragged_batch_multi_chunk(ctx, "two_pass", d, kb, vb)


def test_eight_query_heads_steps_in_two_launches(ctx, chunked):
    F.test_eight_query_heads_decode_steps_and_prefill(ctx)


# -- causal attends as a virtual batch ------------------------------------------------

@pytest.mark.parametrize("mode", ["online", "two_pass"])
def test_prefill_from_a_base_across_chunks(ctx, virtual_batch, chunk_tokens, mode):
    P.test_prefill_from_a_base_across_chunks_and_query_batches(ctx, mode)


@pytest.mark.parametrize("mode", ["online", "two_pass"])
def test_prefill_over_several_launches(ctx, virtual_batch, mode):
    """More queries than one launch of the virtual batch takes (1,024)."""
    from insitu_amd.attention import CompressedAttention
    base, n = 37, 1030
    rng = np.random.default_rng(9)
    k, v = P._random_cache_inputs(rng, base + n)
    c = P._cache(ctx, base + n)
    c.append_rotated(k, v)
    q = rng.integers(-(1 << 22), 1 << 22, size=(n, 32, 64))
    out = CompressedAttention(c).attend_prefill(q, base, mode)[0].cpu().numpy()
    host = Cache(8, base + n, Format())
    host.append_rotated(k, v)
    heads = [host.view(h) for h in range(8)]
    if mode == "online":
        np.testing.assert_array_equal(out, native.decode_steps(q, heads, Format(), base=base))
        return
    for i in (0, 1022, 1023, 1024, 1025, n - 1):
        want = np.concatenate([native.attend_two_pass(q[i, 4 * h:4 * h + 4],
                                                      heads[h].select(slice(0, base + i + 1)), Format())[0]
                               for h in range(8)])
        np.testing.assert_array_equal(out[i], want, err_msg=f"query {i}")


@pytest.mark.parametrize("mode", ["online", "two_pass"])
@pytest.mark.parametrize("kb,vb", [(4, 2), (5, 2)])
def test_one_kv_head_over_several_launches(ctx, virtual_batch, kb, vb, mode):
    """More queries of one KV head than one launch takes: a later launch's queries and outputs lie at
    that head's stride, not at the whole sequence's (5-bit keys: the token loop, launched alike)."""
    from insitu_amd.attention import CompressedAttention
    base, n, h, f = 5, 1030, 6, Format(key_bits=kb, value_bits=vb)
    rng = np.random.default_rng(10)
    k, v = P._random_cache_inputs(rng, base + n)
    c = P._cache(ctx, base + n, kb=kb, vb=vb)
    c.append_rotated(k, v)
    q = rng.integers(-(1 << 22), 1 << 22, size=(n, 4, 64))
    a = CompressedAttention(c)
    out, st = (a.attend_online_batch if mode == "online" else a.attend_causal_batch)(q, h, base)
    host = Cache(8, base + n, f)
    host.append_rotated(k, v)
    kv = host.view(h)
    fn = native.attend_online if mode == "online" else native.attend_two_pass
    for i in range(n):
        np.testing.assert_array_equal(out[i], fn(q[i], kv.select(slice(0, base + i + 1)), f)[0], err_msg=f"query {i}")
    assert st.n_tokens == base + n


@pytest.mark.parametrize("mode", ["online", "two_pass"])
@pytest.mark.parametrize("kb,vb", [(4, 2), (3, 2), (2, 3)])
def test_prefill_is_the_token_loop(ctx, virtual_batch, kb, vb, mode):
    P.test_prefill_is_the_token_loop(ctx, kb, vb, mode)


@pytest.mark.parametrize("softmax", ["online", "two_pass"])
def test_block_prefill_equals_the_decode_loop(ctx, chunked, softmax):
    P.test_block_prefill_equals_the_decode_loop(ctx, softmax)


def test_prefill_of_one_kv_head(ctx, virtual_batch):
    P.test_prefill_group_interface_and_bounds(ctx)


def test_signed_norm_rows(ctx, virtual_batch):
    P.test_signed_norm_edge_rows_on_the_device(ctx)


def test_epoch_wrap_of_each_buffer(ctx, virtual_batch):
    """The first prompt lays the prefill scratch out for 2,600 queries, so that the later ones reach
    its wrap without growing it (which starts its count again)."""
    S.test_epoch_wrap_of_each_buffer_in_either_order(ctx)


@pytest.mark.parametrize("mode", ["online", "two_pass"])
def test_static_array_is_reused(ctx, virtual_batch, chunk_tokens, mode):
    Z.test_static_prefill_equals_the_allocating_prefill_twice(ctx, mode)
