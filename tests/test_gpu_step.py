"""The dense recurrences with one launch per step (scan_step.hip), which serve
gru_scan / gru_scan_forward / gru_scan_backward_triton above 128 hidden units
and every dense recurrence above 1024. Their products follow the persistent
kernels' order, so up to H = 1024 both must agree bit for bit; above, the
oracle checks of test_gpu_tiled.py apply. Sizes sit on the edges of the 16-row,
16-unit and 64-k tiles and on each rows-per-workgroup variant."""

from __future__ import annotations

import ctypes

import pytest
import torch

from gru_qat_amd.configs import Q_INT8_HIDDEN, make_config
from parity_util import log, to_dev

pytestmark = pytest.mark.gpu

OTHER = (0.05, -10, 10)
# (T, B, H): 129 the smallest H; 16 / 17 and 64 / 65 rows; K one past and one short of a chunk; rows of every
# length modulo 4; T H^2 on both sides of the training scans' bound; 32 rows a workgroup (B = 90 x 1000). At
# (2, 250, 1024) the persistent entries take the launches too: it compares the entries, not the kernels (64 rows a
# workgroup: test_step_variants_match_small_batches)
SHAPES = [(13, 1, 129), (25, 1, 129), (11, 16, 130), (24, 17, 131), (7, 65, 257), (3, 17, 191), (4, 65, 257),
          (1, 33, 192), (3, 90, 1000), (2, 250, 1024)]


def _cfg(shape, q_in=None, q_out=None, int8=False):
    cfg = make_config(2 if int8 else 1, shape=shape, seed=3)
    cfg["h_in_quant"], cfg["h_out_quant"] = q_in, q_out
    return cfg


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("q_in,q_out", [(None, None), (Q_INT8_HIDDEN, Q_INT8_HIDDEN), (OTHER, Q_INT8_HIDDEN),
                                        (None, OTHER)])
def test_step_matches_persistent(dev, shape, q_in, q_out):
    import gru_qat_amd.scan as S

    cfg = _cfg(shape, q_in, q_out)
    d = to_dev(cfg, dev)
    T, B, H = shape
    outs, ghs = [], []
    for tiled in (True, False):
        gh = torch.empty((T, B, 3 * H), device=dev)
        outs.append(S._dense_forward("test", d["gi"], d["h0"], d["w"], d["bh"], q_in, q_out, gh_save=gh, tiled=tiled))
        ghs.append(gh)
    plain = S._dense_forward("test", d["gi"], d["h0"], d["w"], d["bh"], q_in, q_out, tiled=True)
    assert torch.equal(outs[0], outs[1]) and torch.equal(ghs[0], ghs[1]) and torch.equal(plain, outs[0])
    dout = torch.randn(outs[0].shape, generator=torch.Generator().manual_seed(5)).to(dev)
    a = S.gru_scan_backward_triton(d["gi"], d["h0"], d["w"], d["bh"], outs[0], dout, h_in_quant=q_in, h_out_quant=q_out)
    b = S.gru_scan_backward_persistent(d["gi"], d["h0"], d["w"], d["bh"], outs[0], dout, h_in_quant=q_in,
                                       h_out_quant=q_out)
    for name, x, y in zip(("dgi", "dh0", "dWh", "dbh"), a, b):
        assert torch.equal(x, y), name


@pytest.mark.parametrize("shape", [(3, 1, 144), (3, 17, 272), (2, 60, 1024), (2, 33, 1040)])
@pytest.mark.parametrize("q_out", [Q_INT8_HIDDEN, None])
def test_step_int8_codes(dev, shape, q_out):
    """Exact integer sums: the persistent int8 kernel's outputs up to H = 1024, and within one level of the
    fp32 products above (a code on a rounding boundary may fall either way)."""
    import gru_qat_amd.scan as S

    cfg = _cfg(shape, Q_INT8_HIDDEN, q_out, int8=True)
    d = to_dev(cfg, dev)
    args = (d["gi"], d["h0"], d["w"], d["bh"], Q_INT8_HIDDEN, q_out)
    a = S._dense_forward("test", *args, tiled=True, int8_codes=True)
    if shape[2] <= 1024:
        assert torch.equal(a, S._dense_forward("test", *args, int8_codes=True))
    else:
        err = (a - S._dense_forward("test", *args, tiled=True)).abs().max().item()
        assert err <= 1.01 / 127, err


def _rows(d, lo, n, dout=None):
    rows = slice(lo, lo + n)
    cut = [d["gi"][:, rows].contiguous(), d["h0"][rows].contiguous()]
    return cut if dout is None else cut + [dout[:, rows].contiguous()]


# 64 rows x 16 units a workgroup forward and 32 x 32 backward, with whole 16-byte rows and with a rest of one float;
# a last workgroup of 47 rows (B = 239) or 8 (B = 200)
@pytest.mark.parametrize("shape", [(2, 239, 1024), (2, 239, 1021), (2, 200, 1001)])
@pytest.mark.parametrize("q_in,q_out", [(None, None), (Q_INT8_HIDDEN, Q_INT8_HIDDEN), (OTHER, Q_INT8_HIDDEN)])
def test_step_variants_match_small_batches(dev, shape, q_in, q_out):
    """The variants of large batches through the barrier-free entries: rows of the first, a middle and the last
    tile equal the same rows as a batch of five, which the persistent kernels run."""
    import gru_qat_amd.scan as S

    cfg = _cfg(shape, q_in, q_out)
    d = to_dev(cfg, dev)
    T, B, H = shape
    dout = torch.randn((T, B, H), generator=torch.Generator().manual_seed(5)).to(dev)
    gh = torch.empty((T, B, 3 * H), device=dev)
    out = S._dense_forward("test", d["gi"], d["h0"], d["w"], d["bh"], q_in, q_out, gh_save=gh, tiled=True)
    plain = S._dense_forward("test", d["gi"], d["h0"], d["w"], d["bh"], q_in, q_out, tiled=True)
    assert torch.equal(out, plain)
    dgi, dh0 = S._dense_backward("test", d["gi"], d["h0"], d["w"], d["bh"], out, dout, q_in, q_out, gh_saved=gh,
                                 tiled=True)[:2]
    for lo in (0, 62, B - 5):
        gi, h0, do = _rows(d, lo, 5, dout)
        gh5 = torch.empty((T, 5, 3 * H), device=dev)
        out5 = S._dense_forward("test", gi, h0, d["w"], d["bh"], q_in, q_out, gh_save=gh5)
        g5 = S._dense_backward("test", gi, h0, d["w"], d["bh"], out5, do, q_in, q_out, gh_saved=gh5)
        for name, x, y in (("out", out, out5), ("gh", gh, gh5), ("dgi", dgi, g5[0]), ("dh0", dh0[None], g5[1][None])):
            assert torch.equal(x[:, lo:lo + 5], y), (name, lo)


# 32 rows x 16 units a workgroup, chunks of 256 codes in pairs: two, four and three of them
@pytest.mark.parametrize("shape", [(2, 225, 512), (2, 239, 1024), (3, 209, 528)])
@pytest.mark.parametrize("q_out", [Q_INT8_HIDDEN, None])
def test_step_int8_large_batches(dev, shape, q_out):
    import gru_qat_amd.scan as S

    d = to_dev(_cfg(shape, Q_INT8_HIDDEN, q_out, int8=True), dev)
    out = S._dense_forward("test", d["gi"], d["h0"], d["w"], d["bh"], Q_INT8_HIDDEN, q_out, tiled=True, int8_codes=True)
    for lo in (0, 30, shape[1] - 5):
        part = S._dense_forward("test", *_rows(d, lo, 5), d["w"], d["bh"], Q_INT8_HIDDEN, q_out, int8_codes=True)
        assert torch.equal(out[:, lo:lo + 5], part), lo


# (11, 48, 1000): launches backward only, its forward is a round short of the rule; the others both ways
@pytest.mark.parametrize("shape", [(11, 48, 1000), (7, 65, 1000), (8, 97, 640), (4, 250, 501), (1, 260, 320)])
@pytest.mark.parametrize("q", [None, Q_INT8_HIDDEN])
def test_large_batches_on_the_persistent_entries(dev, shape, q):
    """gru_scan_persistent's batches that run with a launch per step: every row equals the same row of a
    batch small enough for the persistent kernel, forward (fp32 and int8 codes), gh and gradients."""
    import gru_qat_amd.scan as S

    cfg = _cfg(shape, q, q, int8=q is not None)
    d = to_dev(cfg, dev)
    T, B, H = shape
    n = 5

    def run(gi, h0, dout, codes):
        gh = None if codes else torch.empty((T, gi.shape[1], 3 * H), device=dev)
        out = S._dense_forward("test", gi, h0, d["w"], d["bh"], q, q, gh_save=gh, int8_codes=codes)
        if codes:
            return [out]
        g = S._dense_backward("test", gi, h0, d["w"], d["bh"], out, dout, q, q, gh_saved=gh)
        return [out, gh, g[0], g[1][None]]

    dout = torch.randn((T, B, H), generator=torch.Generator().manual_seed(5)).to(dev)
    for codes in (False, True) if q is not None and H % 16 == 0 else (False,):
        whole = run(d["gi"], d["h0"], dout, codes)
        for lo in (0, B - n):
            rows = slice(lo, lo + n)
            part = run(d["gi"][:, rows].contiguous(), d["h0"][rows].contiguous(), dout[:, rows].contiguous(), codes)
            for x, y in zip(whole, part):
                assert torch.equal(x[:, rows], y), (codes, lo)


def _raw(dev, name, gi, h0, w, bh, out, T, B, H, sg, so, sh0, q=None, codes=None):
    from gru_qat_amd import _lib

    lib = _lib.load()
    a = _lib.GsArgs(gi.data_ptr(), h0.data_ptr(), w.data_ptr(), None, bh.data_ptr(), out.data_ptr(), None, 0, None, T,
                    B, H, *sg, sh0, *so, 0, 0, 0, 0, _lib.make_quant(q, "q"), _lib.make_quant(q, "q"), None)
    extra = [] if codes is None else [ctypes.c_void_p(c.data_ptr()) for c in codes]
    rc = getattr(lib, name)(ctypes.byref(a), *extra, ctypes.c_void_p(_lib.current_stream_handle(dev)))
    _lib.raise_for(rc, lib)
    torch.cuda.synchronize(dev)


@pytest.mark.parametrize("pad", [1, 4])
def test_step_strided_and_unaligned(dev, pad):
    """Padded rows of gi, h0 and out, and bases off 16 bytes (pad 1), give the contiguous call's outputs."""
    T, B, H = 3, 19, 146
    cfg = _cfg((T, B, H))
    d = to_dev(cfg, dev)
    ref = torch.empty((T, B, H), device=dev)
    _raw(dev, "gs_dense_fwd_tiled", d["gi"], d["h0"], d["w"], d["bh"], ref, T, B, H, (B * 3 * H, 3 * H), (B * H, H), H)
    gi = torch.full((T, B + 1, 3 * H + pad), float("nan"), device=dev)
    gi[:, :B, pad:] = d["gi"]
    h0 = torch.full((B, H + pad), float("nan"), device=dev)
    h0[:, pad:] = d["h0"]
    w = torch.full((3 * H * H + pad,), float("nan"), device=dev)
    w[pad:] = d["w"].reshape(-1)
    out = torch.full((T, B + 2, H + pad), 7.0, device=dev)
    _raw(dev, "gs_dense_fwd_tiled", gi[0, 0, pad:], h0[0, pad:], w[pad:], d["bh"], out[0, 0, pad:], T, B, H,
         gi.stride()[:2], out.stride()[:2], h0.stride(0))
    assert torch.equal(out[:, :B, pad:], ref)
    assert (out[:, :, :pad] == 7.0).all() and (out[:, B:] == 7.0).all()


def test_step_in_place_state(dev):
    """out on top of h0 (a streaming state updated in place) keeps running one batch tile per workgroup."""
    T, B, H = 1, 37, 512
    cfg = _cfg((T, B, H))
    d = to_dev(cfg, dev)
    ref = torch.empty((T, B, H), device=dev)
    _raw(dev, "gs_dense_fwd_tiled", d["gi"], d["h0"], d["w"], d["bh"], ref, T, B, H, (B * 3 * H, 3 * H), (B * H, H), H)
    state = d["h0"].clone()
    _raw(dev, "gs_dense_fwd_tiled", d["gi"], state, d["w"], d["bh"], state, T, B, H, (B * 3 * H, 3 * H), (B * H, H), H)
    log(f"[step] in place: {int((state != ref[0]).sum())} elements differ")
    assert torch.equal(state, ref[0])


@pytest.mark.parametrize("B,H", [(19, 144), (209, 528)])  # 16 and 32 rows a workgroup
@pytest.mark.parametrize("pad", [1, 4])
def test_step_int8_strided_and_unaligned(dev, B, H, pad):
    """Padded rows, and h0 and out off 16 bytes (pad 1), with int8 codes."""
    from gru_qat_amd import _lib

    T, q = 3, Q_INT8_HIDDEN
    d = to_dev(_cfg((T, B, H), q, q, int8=True), dev)
    codes = _lib.weight_codes(d["w"])
    assert codes is not None
    ref = torch.empty((T, B, H), device=dev)
    name = "gs_dense_fwd_tiled_i8w"
    _raw(dev, name, d["gi"], d["h0"], d["w"], d["bh"], ref, T, B, H, (B * 3 * H, 3 * H), (B * H, H), H, q, codes)
    h0 = torch.full((B, H + pad), float("nan"), device=dev)
    h0[:, pad:] = d["h0"]
    out = torch.full((T, B + 2, H + pad), 7.0, device=dev)
    _raw(dev, name, d["gi"], h0[0, pad:], d["w"], d["bh"], out[0, 0, pad:], T, B, H, (B * 3 * H, 3 * H),
         out.stride()[:2], h0.stride(0), q, codes)
    assert torch.equal(out[:, :B, pad:], ref)
    assert (out[:, :, :pad] == 7.0).all() and (out[:, B:] == 7.0).all()


@pytest.mark.parametrize("H", [512, 1040])
@pytest.mark.parametrize("int8", [False, True])
def test_step_in_place_state_one_cu_kernels(dev, H, int8):
    """out on top of h0 with int8 codes and above H = 1024: the batch-tiled kernels, which such calls keep."""
    from gru_qat_amd import _lib

    T, B, q = 1, 37, Q_INT8_HIDDEN if int8 else None
    d = to_dev(_cfg((T, B, H), q, q, int8=int8), dev)
    name, codes = ("gs_dense_fwd_tiled_i8w", _lib.weight_codes(d["w"])) if int8 else ("gs_dense_fwd_tiled", None)
    args = (T, B, H, (B * 3 * H, 3 * H), (B * H, H), H, q, codes)
    ref = torch.empty((T, B, H), device=dev)
    _raw(dev, name, d["gi"], d["h0"], d["w"], d["bh"], ref, *args)
    state = d["h0"].clone()
    _raw(dev, name, d["gi"], state, d["w"], d["bh"], state, *args)
    assert torch.equal(state, ref[0])
