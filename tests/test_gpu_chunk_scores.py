"""The chunked attend's matrix-core scores at their edges: every key width, head dimension and
chunk build, context lengths around the tiles and the halves of a wave, and query values at the
ends of int32, against the token-by-token kernel and, in two-pass mode, oracle/c."""

import numpy as np
import pytest
import torch

from oracle import native
from oracle.quantize import Format

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunk_tokens", [512, 1024])
@pytest.mark.parametrize("d,kb,vb", [(64, 2, 1), (64, 3, 2), (64, 4, 2), (128, 2, 2), (128, 3, 3), (128, 4, 2)])
def test_scores_equal_the_token_by_token_kernel(ctx, d, kb, vb, chunk_tokens):
    from insitu_amd import CompressedAttention, CompressedCache, QuantConfig
    lens = [1, 15, 17, 31, 33, 63, 65, 127, 129, 511, 513, 1023, 1025, 1100]
    cache = CompressedCache(2, d, max(lens), QuantConfig(key_bits=kb, value_bits=vb), batch=len(lens), n_q_heads=8,
                            chunk_tokens=chunk_tokens, ctx=ctx)
    cache.pin_kernel("chunked")
    rng = np.random.default_rng(d + kb)

    def rows(n, heads):
        x = np.rint(rng.standard_normal((n, heads, d)) * 65536)
        return torch.from_numpy(x.astype(np.int32)).to(ctx.torch_device)

    for b, n in enumerate(lens):
        cache.append_rotated(rows(n, 2), rows(n, 2), seq=b)
    attn = CompressedAttention(cache)
    q = rows(len(lens), 8)
    q[0, 0, :4] = torch.tensor([2**31 - 1, -2**31, 2**31 - 1 - 0x808080, 2**30], dtype=torch.int32)
    q[1, 1, :3] = torch.tensor([2**31 - 1 - 0x808080, -2**31, 2**30], dtype=torch.int32)
    q[2] = 2**26
    q[3] = -2**26
    for scale in (1, 8):                    # peaked and flatter weights
        qs = torch.div(q, scale, rounding_mode="floor").to(torch.int32)
        got = attn.attend(qs, "online", stats=False)[0]
        want = attn.attend(qs, "serial", stats=False)[0]
        assert torch.equal(got, want)
        out = attn.attend(qs, "two_pass", stats=False)[0].cpu().numpy()
        q_np = qs.cpu().numpy()
        for b in range(len(lens)):
            for h in range(2):
                kv = cache.view(h, seq=b).host()
                want = native.attend_two_pass(q_np[b, 4 * h:4 * h + 4], kv, Format(d=d, key_bits=kb, value_bits=vb))[0]
                np.testing.assert_array_equal(out[b, 4 * h:4 * h + 4], want, err_msg=f"{lens[b]} rows, head {h}")
