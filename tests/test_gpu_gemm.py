"""The fp32 products behind the projections, at the edges of their tiles: each
layout (NT: gi, NN: dx, TN: dW) with 64 x 64 and with 128 x 128 tiles, 16-byte
and single-word loads, remainders in every dimension, rows off 16-byte boundaries and rows too far apart for 32-bit offsets, against the same
products in float64."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

U32 = 2.0 ** -24


def _close(name, got, a, b, bias=None):
    """got = a b within the bound of a float32 sum in any order: K roundings of
    at most the sum of the magnitudes each, here as |a| |b| K u (and one for
    the bias), in float64."""
    a, b = a.double(), b.double()
    ref, mag = a @ b, a.abs() @ b.abs()
    if bias is not None:
        ref, mag = ref + bias.double(), mag + bias.double().abs()
    bound = (a.shape[1] + 1) * U32 * mag
    bad = (got.double() - ref).abs() > bound
    assert not bad.any(), f"{name}: {int(bad.sum())} of {bad.numel()} past the bound"


@pytest.mark.parametrize("M,N,K", [
    (1, 3, 1), (2, 3, 4), (64, 66, 31), (65, 63, 32), (63, 129, 33), (130, 192, 64), (257, 60, 100),
    (67, 5, 33), (5, 66, 35), (66, 7, 6),
    (700, 63, 1027),        # K splits of dW and dx with a short last one
    (8180, 2046, 2046),     # 128 x 128 tiles in all three layouts, single words
    (8180, 2040, 2044),     # the same in 16-byte loads
])
@pytest.mark.parametrize("shift", [0, 1])
def test_products(dev, M, N, K, shift):
    import gru_qat_amd as G

    print(f"[gemm] M={M} N={N} K={K} shift={shift}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)

    def rows(n, k):  # rows of k + 3 * shift floats from the shift-th float on
        full = torch.randn(n, k + 3 * shift, generator=g).to(dev)
        return full[:, shift:shift + k]

    x, dgi = rows(M, K).requires_grad_(True), rows(M, N)
    w = (torch.randn(N, K, generator=g) / K ** 0.5).to(dev).requires_grad_(True)
    b = torch.randn(N, generator=g).to(dev).requires_grad_(True)
    gi = G.input_projection(x, w, b)
    dx, dw = torch.autograd.grad(gi, [x, w], dgi)
    with torch.no_grad():
        _close("gi", gi, x, w.t(), b)
        _close("dx", dx, dgi, w)
        _close("dw", dw, dgi.t(), x)


def test_far_rows(dev):
    """Rows 2^24 + 4 floats apart: a tile's offsets do not fit 32 bits."""
    import gru_qat_amd as G

    M, N, K, ld = 6, 9, 37, (1 << 24) + 4
    store = torch.zeros((M - 1) * ld + K, device=dev)
    x = store.as_strided((M, K), (ld, 1))
    g = torch.Generator().manual_seed(0)
    x.copy_(torch.randn(M, K, generator=g))
    x.requires_grad_(True)
    w = torch.randn(N, K, generator=g).to(dev).requires_grad_(True)
    dgi = torch.randn(M, N, generator=g).to(dev)
    gi = G.input_projection(x, w, None)
    dw, = torch.autograd.grad(gi, [w], dgi)
    with torch.no_grad():
        _close("gi", gi, x, w.t())
        _close("dw", dw, dgi.t(), x)
