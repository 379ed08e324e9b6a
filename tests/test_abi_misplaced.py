"""C ABI: arguments that an entry point must not take silently, rejected before any HIP call (nothing is launched)."""

import ctypes as ct

import pytest

from mamformer_amd import _lib
from tests.test_abi import _good_bwd, _good_ssd, _good_ssu, _rc


def _ref(a):
    """The reference form of the scan arguments: one group, a rate per state, a step per channel."""
    a.ngroups, a.B_stride_l, a.C_stride_l = 1, a.dstate, a.dstate
    a.dt_stride_l = a.nheads * a.headdim
    a.dt_stride_b = a.seqlen * a.dt_stride_l
    a.flags |= _lib.MH_A_PER_STATE | _lib.MH_DT_PER_CHANNEL
    return a


def test_log_rates_belong_to_the_reference_scan():
    n = ct.c_size_t()
    a = _ref(_good_ssd())
    a.flags |= _lib.MH_A_LOG
    assert _rc("mh_ssd_ref_scan_workspace_bytes", ct.byref(a), 1, ct.byref(n)) == 0
    a = _good_ssd()
    a.flags |= _lib.MH_A_LOG
    cl = ct.c_int64()
    for call in (lambda: _rc("mh_ssd_workspace_bytes", ct.byref(a), ct.byref(n)),
                 lambda: _rc("mh_ssd_chunk_len", ct.byref(a), ct.byref(cl)),
                 lambda: _rc("mh_ssd_chunk_scan_fwd", ct.byref(a), None),
                 lambda: _rc("mh_ssd_chunk_scan_fwd_noalloc", ct.byref(a), None)):
        assert call() == -6 and b"MH_A_LOG" in _lib.lib().mh_last_error()
    b = _good_bwd()
    b.fwd.flags |= _lib.MH_A_LOG
    assert _rc("mh_ssd_bwd_workspace_bytes", ct.byref(b), ct.byref(n)) == -6


@pytest.mark.parametrize("flags", [0, _lib.MH_A_PER_STATE | _lib.MH_DT_PER_CHANNEL])
def test_state_update_refuses_log_rates(flags):
    u = _good_ssu()
    u.dt_stride_b = 8 * 64
    u.flags = flags | _lib.MH_A_LOG
    assert _rc("mh_ssd_state_update", ct.byref(u), None) == -6
    assert b"MH_A_LOG" in _lib.lib().mh_last_error()
