"""What the order loops refuse before they launch anything: plans whose arrays
or sizes a kernel would read past.  The addresses are never followed."""
import ctypes

import pytest

from sparrowpy_amd import _hip

S = _hip.ExchangePlanStruct
SOMEWHERE = 1 << 20


def _plan(kind, **changed):
    st = S(kind=kind, P=2, D=3, B=1, Vd=2, max_lag=1, max_groups=1)
    for name in S.ARRAYS:
        setattr(st, name, SOMEWHERE)
    for name, value in changed.items():
        setattr(st, name, value)
    return st


def _codes(st):
    """The codes of the forward loops and of the plan's adjoint segment."""
    lib = _hip.lib(require_gpu=False)
    a = ctypes.addressof(st)
    bufs = (ctypes.c_void_p * 2)(SOMEWHERE, 2 * SOMEWHERE)
    p = [SOMEWHERE * k for k in range(1, 16)]
    codes = [lib.spr_exchange_orders(a, 5, 2, 5, p[0], p[1], 343., 1., p[2],
                                     p[3], bufs, p[4], p[5], p[6], None),
             lib.spr_exchange_sum(a, 5, 2, 5, p[0], p[1], 343., 1., p[2],
                                  p[3], p[4], p[5], p[6], None)]
    if st.kind == S.DS:
        codes.append(lib.spr_adjoint_segment_ds(a, 5, 0, 2, 5, bufs, *p[:13],
                                                None))
    else:
        codes.append(lib.spr_adjoint_segment_grouped(a, 5, 0, 2, 5, bufs,
                                                     bufs, *p[:10], None))
    return codes


@pytest.mark.parametrize("kind,changed", [
    (S.DS, dict(grp_start=None)), (S.DS, dict(dscal=None)),
    (S.DS, dict(max_groups=0)), (S.GROUPED, dict(max_groups=0)),
    (S.GROUPED, dict(max_groups=-3)), (S.GROUPED, dict(rtab=None)),
    (S.DS, dict(grp_ptr=None))])
def test_incomplete_plans_are_refused(kind, changed):
    assert _codes(_plan(kind, **changed)) == [-1] * 3   # SPR_ERR_ARG
