"""The observer scan's one launch per step (observe.hip) at the edges of its
tiles: 16 units, 16 or 32 rows, K splits of 32-k slices, row ends of every
length, more partials than a wave's first loads, one quantizer in both places;
and its three launches per step for large batches. Checked step by step from the
kernel's own previous output, as in test_gpu_observe.py, and the two forms
against each other."""

from __future__ import annotations

import ctypes

import pytest
import torch

import gru_qat_amd as G
from oracle import gru_oracle as O
from parity_util import to_dev
from test_gpu_observe import _cfg, _codes_match, _frozen, _quant, _run, _teacher_forced

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(3, 2, 1), (3, 2, 3), (3, 17, 6), (3, 15, 33), (2, 33, 127), (2, 16, 130), (2, 3, 517),
                                   (2, 280, 257),     # 32 rows a workgroup
                                   (2, 1500, 256),    # three rounds of workgroups, 752 partials
                                   (2, 2200, 256)])   # four: three launches a step
@pytest.mark.parametrize("mode,symmetric", [("min_max", True), ("dynamic", False)])
def test_observe_step_edges(dev, shape, mode, symmetric):
    cfg = _cfg(1, shape)
    q_in, q_out = _quant(mode, symmetric).to(dev), _quant(mode, symmetric).to(dev)
    out, trace = _run(cfg, dev, q_in, q_out)
    out, trace = out.cpu(), trace.cpu()
    st_in, st_out = O.ObserverState(mode, symmetric=symmetric), O.ObserverState(mode, symmetric=symmetric)
    pre, sc = _teacher_forced(cfg, out, st_in, st_out)
    assert torch.equal(trace[:, :2], sc[:, :2])
    assert torch.allclose(trace[:, 2], sc[:, 2], rtol=1e-5, atol=0)
    for t in range(shape[0]):
        _codes_match(out[t], pre[t], float(trace[t, 2]), float(trace[t, 3]), q_out.qmin, q_out.qmax)
    if mode == "min_max":
        assert torch.equal(q_in.observer_stats.cpu()[:2], torch.stack([st_in.running_min, st_in.running_max]))


@pytest.mark.parametrize("idx,shape", [(1, (4, 5, 96)), (0, (4, 5, 96))])
def test_observe_one_quantizer_in_both_places(dev, idx, shape):
    cfg = _cfg(idx, shape)
    q = _quant("min_max", True).to(dev)
    out, _ = _run(cfg, dev, q, q)
    st = O.ObserverState("min_max")
    _teacher_forced(cfg, out.cpu(), st, st)
    assert torch.allclose(q.observer_stats.cpu()[:2], torch.stack([st.running_min, st.running_max]), rtol=1e-5)


@pytest.mark.parametrize("idx", [0, 1])
@pytest.mark.parametrize("which", ["in", "out"])
def test_observe_one_side_off(dev, idx, which):
    cfg = _cfg(idx, (4, 19, 70))
    q = _quant("min_max", True).to(dev)
    out, trace = _run(cfg, dev, q if which == "in" else None, q if which == "out" else None)
    out = out.cpu()
    c = {k: (v.cpu() if isinstance(v, torch.Tensor) else v) for k, v in cfg.items()}
    gh_fn, st = O.gh_fn_for(c), O.ObserverState("min_max")
    for t in range(out.shape[0]):
        h = c["h0"] if t == 0 else out[t - 1]
        hq = O.observer_forward(st, h)[0] if which == "in" else h
        pre = O.gru_step(c["gi"][t], h, gh_fn(hq))
        if which == "in":
            assert (out[t] - pre).abs().max() <= 1e-5
        else:
            s = O.observer_forward(st, pre)[1][0]
            assert abs(float(trace[t, 2]) - s) <= 1e-5 * s
            _codes_match(out[t], pre, float(trace[t, 2]), 0.0, -127, 127)
    assert torch.allclose(q.observer_stats.cpu()[:2], torch.stack([st.running_min, st.running_max]), rtol=1e-5)


def _observe_raw(dev, kind, gi, h0, w, bh, q_in, q_out):
    """gs_observe_scan on device tensors with the C ABI's own observers."""
    from gru_qat_amd import _lib

    lib = _lib.load()
    T, B, H3 = gi.shape
    out = torch.empty((T, B, H3 // 3), device=dev)
    a = _lib.GsObserveArgs(kind=kind, gi=gi.data_ptr(), h0=h0.data_ptr(), w=w.data_ptr(), bh=bh.data_ptr(),
                           out=out.data_ptr(), T=T, B=B, H=H3 // 3, sg_t=gi.stride(0), sg_b=gi.stride(1),
                           sh0_b=h0.stride(0), so_t=out.stride(0), so_b=out.stride(1), q_in=q_in, q_out=q_out)
    need = lib.gs_observe_scan_scratch_bytes(ctypes.byref(a))
    _lib.raise_for(min(need, 0), lib)
    scratch = torch.empty(int(need), dtype=torch.uint8, device=dev)
    a.scratch, a.scratch_bytes = scratch.data_ptr(), scratch.numel()
    _lib.raise_for(lib.gs_observe_scan(ctypes.byref(a), ctypes.c_void_p(_lib.current_stream_handle(dev))), lib)
    torch.cuda.synchronize(dev)
    return out


@pytest.mark.parametrize("idx", [0, 1])
def test_observe_shared_stats_pointer_with_other_modes(dev, idx):
    """A dynamic q_out keeps no statistics, so a stats pointer that it shares with a min_max q_in is q_in's alone."""
    from gru_qat_amd import _lib

    cfg = _cfg(idx, (4, 5, 96))
    d = to_dev(cfg, dev)
    got = []
    for shared in (False, True):
        stats = torch.tensor([float("inf"), float("-inf"), 0.0], device=dev)
        q_in = _lib.GsObserver(_lib.OBS_MIN_MAX, 1, -127, 127, 1.0, 0.0, stats.data_ptr())
        q_out = _lib.GsObserver(_lib.OBS_DYNAMIC, 1, -127, 127, 1.0, 0.0, stats.data_ptr() if shared else None)
        kind = _lib.KIND_DIAGONAL if idx == 0 else _lib.KIND_DENSE
        got.append((_observe_raw(dev, kind, d["gi"], d["h0"], d["w"], d["bh"], q_in, q_out), stats))
    assert torch.equal(got[0][0], got[1][0])
    assert torch.equal(got[0][1], got[1][1]), (got[0][1].tolist(), got[1][1].tolist())


@pytest.mark.parametrize("idx", [0, 1])
@pytest.mark.parametrize("mode", ["frozen", "dynamic"])
def test_observe_codes_past_24_bits(dev, idx, mode):
    """Ranges past the bound of the division-free quotient take the IEEE one: out[0], which the launch of step 1
    quantizes, is fake_quant_ste's of the pre-quant state bit for bit."""
    from gru_qat_amd import _lib

    T, B, H = 2, 37, 64
    cfg = _cfg(idx, (T, B, H))
    d = to_dev(cfg, dev)
    args = (_lib.KIND_DIAGONAL if idx == 0 else _lib.KIND_DENSE, d["gi"], d["h0"], d["w"], d["bh"])
    off = _lib.GsObserver(_lib.OBS_OFF, 1, 0, 1, 1.0, 0.0, None)
    pre = _observe_raw(dev, *args, off, off)[0].cpu()
    lim = 2 ** 30
    s = torch.tensor(1e-9) if mode == "frozen" else pre.abs().max().clamp(min=1e-8) / torch.tensor(float(lim))
    q_out = _lib.GsObserver(_lib.OBS_FROZEN if mode == "frozen" else _lib.OBS_DYNAMIC, 1, -lim, lim, 1e-9, 0.0, None)
    out = _observe_raw(dev, *args, off, q_out)[0].cpu()
    ref = torch.round(pre / s).clamp(-lim, lim) * s
    assert torch.equal(out, ref), f"{int((out != ref).sum())} of {ref.numel()} differ"


@pytest.mark.parametrize("shape", [(3, 2100, 100), (2, 8200, 64), (2, 260, 640), (3, 8200, 33), (2, 70, 3072)])
@pytest.mark.parametrize("q_in,q_out", [(None, None), (0.01, 0.01), (0.02, None), (None, 0.03)])
def test_observe_three_launches_match_one(dev, shape, q_in, q_out):
    """Rows of a batch that takes three launches a step equal the same rows alone, which take one."""
    cfg = _cfg(1, shape)
    qs = [None if s is None else _frozen(s) for s in (q_in, q_out)]
    whole, _ = _run(cfg, dev, *qs)
    for lo in (0, shape[1] - 7):
        part = dict(cfg, gi=cfg["gi"][:, lo:lo + 7].contiguous(), h0=cfg["h0"][lo:lo + 7].contiguous(), B=7)
        assert torch.equal(whole[:, lo:lo + 7], _run(part, dev, *qs)[0]), lo


def test_observe_batch_past_the_grid(dev):
    """32-row tiles of 2097121 rows are one more than a grid's second dimension holds."""
    T, B, H = 2, 32 * 65535 + 1, 2
    cfg = _cfg(1, (T, B, H))
    q = _quant("min_max", True).to(dev)
    out, trace = _run(cfg, dev, q, None)
    for lo in (0, B - 7):
        part = dict(cfg, gi=cfg["gi"][:, lo:lo + 7].contiguous(), h0=cfg["h0"][lo:lo + 7].contiguous(), B=7)
        for t in range(T):  # one step at the whole batch's scale
            step = dict(part, gi=part["gi"][t:t + 1], h0=part["h0"] if t == 0 else out[t - 1, lo:lo + 7].cpu(), T=1)
            assert torch.equal(out[t, lo:lo + 7], _run(step, dev, _frozen(float(trace[t, 0])), None)[0][0])
    scale = torch.stack([cfg["h0"].abs().max(), out[0].abs().max().cpu()]) / 127.0
    assert torch.equal(trace[:, 0].cpu(), scale)
