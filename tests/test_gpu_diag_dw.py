"""The diagonal input map's weight gradient (column sums of dgi * x over the
rows) at the edges of its chunks of 256 rows, its batches of 128 and its 64
columns, against float64 within the bound of a float32 sum in any order."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 15, 17, 112, 113, 127, 129, 255, 256, 257, 700])
@pytest.mark.parametrize("H", [1, 21, 22, 64, 129])
def test_diagonal_weight_gradient(dev, M, H):
    import gru_qat_amd as G

    g = torch.Generator().manual_seed(1000 * M + H)
    x = torch.randn(M, 1, H, generator=g).to(dev)
    W = torch.randn(3, H, generator=g).to(dev).requires_grad_(True)
    dgi = torch.randn(M, 1, 3 * H, generator=g).to(dev)
    gi = G.structured_input_projection(x, "diagonal", W, None)
    dw, = torch.autograd.grad(gi, [W], dgi)
    terms = (dgi.double() * x.double().repeat(1, 1, 3)).reshape(M, 3 * H)
    bound = (M + 1) * 2.0 ** -24 * terms.abs().sum(0)
    assert ((dw.double().reshape(-1) - terms.sum(0)).abs() <= bound).all()
