"""The prompt's projections on the matrix cores at the edges of their tiles: token counts around 32
and 64, output rows and channels that no tile divides, both input types, with and without a bias, and
rows that the kernel does not take (misaligned, channels not in eights). Against the float64 sum of
the fp16 products, to the bound of an fp32 sum of in_f exact products in any order and the bias."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(y, w, x16, bias):
    w64, x64 = w.astype(np.float64), x16.astype(np.float64)
    exact, mag = x64 @ w64.T, np.abs(x64) @ np.abs(w64).T
    if bias is not None:
        exact, mag = exact + bias, mag + np.abs(bias)
    assert (np.abs(y - exact) <= 2 * (w.shape[1] + 1) * 2.0**-24 * mag + 1e-30).all()


@pytest.mark.parametrize("n", [5, 31, 33, 64, 65, 333])
@pytest.mark.parametrize("out_f,in_f,shift", [(3072, 2048, 0), (37, 8, 0), (66, 136, 0), (128, 130, 0), (64, 256, 1)])
@pytest.mark.parametrize("biased", [False, True])
def test_projection_tiles(ctx, n, out_f, in_f, shift, biased):
    from insitu_amd import _lib
    from insitu_amd.runtime import ptr
    rng = np.random.default_rng(n + out_f)
    dev = ctx.torch_device
    w = (rng.standard_normal((out_f, in_f)) / np.sqrt(in_f)).astype(np.float16)
    wd = torch.from_numpy(w.view(np.int16)).to(dev)
    b = rng.standard_normal(out_f).astype(np.float32) if biased else None
    bd = torch.from_numpy(b).to(dev) if biased else None

    def placed(a):                          # `shift` values past a 16-byte boundary
        t = torch.zeros(a.size + shift, dtype=torch.from_numpy(a).dtype, device=dev)
        t[shift:] = torch.from_numpy(a.reshape(-1)).to(dev)
        return t[shift:]

    bias = ptr(bd) if biased else None
    y = torch.empty((n, out_f), dtype=torch.float32, device=dev)
    x = rng.standard_normal((n, in_f)).astype(np.float32)
    xd = placed(x)
    _lib.check(ctx.lib.insitu_project(ctx.handle, ptr(wd), out_f, in_f, ptr(xd), n, bias, ptr(y)))
    _check(y.cpu().numpy().astype(np.float64), w, x.astype(np.float16), b)
    for frac in (16, 12):
        o = np.rint(rng.standard_normal((n, in_f)) * 2.0**frac).astype(np.int32)
        od = placed(o)
        _lib.check(ctx.lib.insitu_output_projection(ctx.handle, ptr(od), n, in_f, frac, ptr(wd), out_f, bias, ptr(y)))
        _check(y.cpu().numpy().astype(np.float64), w, (o.astype(np.float64) / 2.0**frac).astype(np.float16), b)


@pytest.mark.parametrize("biased", [False, True])
def test_large_tiles(ctx, biased):
    """64 x 64 tiles (264 workgroups) with remainders of tokens, outputs and channels."""
    test_projection_tiles(ctx, 700, 1500, 1000, 0, biased)
