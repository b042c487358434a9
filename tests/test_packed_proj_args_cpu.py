"""The projections pack their argument structures with one struct call; the
bytes must be those of the ctypes structures (the C layout) for the same
values."""

import ctypes

import pytest

from gru_qat_amd import _lib

Q = (1, 0.25, -7, 9)
OFF = _lib._QOFF


def _quants(*qs):
    return [_lib.GsQuant(*q) for q in qs]


@pytest.mark.parametrize("packer,ctype,build", [
    (_lib.PROJ_ARGS, _lib.GsProjArgs, lambda: ((*range(1, 13), *Q, *OFF, 13, 14),
                                               (*range(1, 13), *_quants(Q, OFF), 13, 14))),
    (_lib.PROJ_BWD_ARGS, _lib.GsProjBwdArgs, lambda: ((*range(1, 16), *Q, 16, 17, *OFF),
                                                      (*range(1, 16), *_quants(Q), 16, 17, *_quants(OFF)))),
    (_lib.SPROJ_ARGS, _lib.GsSProjArgs, lambda: ((2, *range(1, 18), *Q, *OFF, *Q, *OFF), (2, *range(1, 18)))),
    (_lib.SPROJ_BWD_ARGS, _lib.GsSProjBwdArgs, lambda: ((2, *range(1, 21), *Q, *OFF, *Q, *OFF), (2, *range(1, 21)))),
], ids=["proj", "proj_bwd", "sproj", "sproj_bwd"])
def test_packed_projection_args_match_the_ctypes_layout(packer, ctype, build):
    fields, values = build()
    a = ctype(*values)
    if hasattr(a, "q_out"):
        a.q_x = _lib.GsQuant(*Q)
        for g, q in enumerate((OFF, Q, OFF)):
            a.q_out[g] = _lib.GsOQuant(*q)
    assert packer.size == ctypes.sizeof(ctype)
    assert packer.pack(*fields) == bytes(a)


def test_quant_fields_match_the_ctypes_fields():
    for bounds in ((-127, 127), (-2**31, 2**31 - 1), (0, 2**32 - 1), (-2**33, 2**31)):  # past 32 bits: wrapped alike
        f = _lib.quant_fields(1, 0.1, *bounds)
        q = _lib.GsQuant(1, 0.1, *bounds)
        assert (f[0], f[2], f[3]) == (q.enabled, q.qmin, q.qmax)
    assert _lib.frozen_fields(None) == OFF
    assert _lib.frozen_fields((0.25, -7, 9)) == Q


def test_size_queries_on_packed_args():
    lib = _lib.load()
    rest = (64, 96, 32, 32, 96, 32, *OFF, 0, 0, *OFF)
    n = _lib.raw_size(lib, "gs_input_proj_bwd_workspace_bytes", _lib.PROJ_BWD_ARGS.pack(*([4096] * 7), 0, 0, *rest))
    a = _lib.GsProjBwdArgs(*([4096] * 7), 0, 0, 64, 96, 32, 32, 96, 32, *_quants(OFF), 0, 0, *_quants(OFF))
    assert n == lib.gs_input_proj_bwd_workspace_bytes(ctypes.byref(a)) >= 0
    with pytest.raises(ValueError):
        _lib.raw_size(lib, "gs_input_proj_bwd_workspace_bytes",
                      _lib.PROJ_BWD_ARGS.pack(*([4096] * 7), 0, 0, 0, *rest[1:]))


@pytest.mark.parametrize("M,N,I", [(1, 3, 1), (64, 96, 32), (1650, 1503, 301), (4282, 5787, 1929)])
def test_projection_backward_workspace_kept_by_size(M, N, I):
    """What the backward keeps per size is the query's answer for its call, quantized or not."""
    from gru_qat_amd.input_proj import _bwd_workspace_bytes

    for q in (OFF, Q):
        a = _lib.GsProjBwdArgs(*([4096] * 7), 0, 0, M, N, I, I + 5, N + 7, I, *_quants(q), 4096, 4096, *_quants(q))
        need = _lib.load().gs_input_proj_bwd_workspace_bytes(ctypes.byref(a))
        assert _bwd_workspace_bytes(M, N, I) == max(need, 256)
    with pytest.raises(ValueError):
        _bwd_workspace_bytes(0, N, I)
