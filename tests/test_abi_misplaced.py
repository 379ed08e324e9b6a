"""C ABI: arguments that an entry point must not take silently, rejected before any HIP call (nothing is launched)."""

import ctypes as ct

import pytest

from mamformer_amd import _lib
from tests.test_abi import _good_bwd, _good_ssd, _good_ssu, _good_step, _rc


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


STATE = 2 * 4 * 128 * 128 * 4                          # bytes of _good_step's state
Z = 2 * 4 * 128 * 4


@pytest.mark.parametrize("state_out,z_out", [
    ("s+16", None), ("s-16", None), (f"s+{STATE - 16}", None), ("z", None), (f"z-{STATE - 16}", None),
    (None, "z+4"), (None, f"z-{Z - 4}"), (None, "s"), (None, f"s+{STATE - 4}"), ("s", "s+64"), ("z", "z"),
    ("n", "n"), ("n", f"n+{STATE - 4}"), ("s", f"z+{Z - 4}"),
])
def test_kda_step_refuses_overlapping_outputs(state_out, z_out):
    a = _good_step()
    at = {"s": 1 << 24, "z": 1 << 25, "n": 1 << 26}     # state, z, a buffer of its own
    a.state, a.z = at["s"], at["z"]
    p = [None if e is None else eval(e, {}, at) for e in (state_out, z_out)]
    assert _rc("mh_kda_recurrent_step_to", ct.byref(a), *p, None) == -4
    assert b"overlap" in _lib.lib().mh_last_error()


def _good_layer_step(width=4, rows=3):
    b, D, H, P, N = 2, 64, 1, 64, 128
    fake = 4096
    a = _lib.LayerStepArgs()
    a.batch, a.d_model, a.nheads, a.headdim, a.dstate, a.ngroups, a.dt_rank, a.width = b, D, H, P, N, 1, 2, width
    for f in ("u", "in_w", "conv_w", "dt_w0", "dt_w1", "B_w", "C_w", "out_w", "A_log", "dt_bias", "D", "out"):
        setattr(a, f, fake)
    a.u_stride_b = D
    a.state_in, a.state_out = 1 << 20, 1 << 22
    a.conv_state, a.conv_out = 1 << 23, 1 << 24
    a.conv_state_len, a.conv_state_stride_l, a.conv_state_stride_b = rows, H * P, rows * H * P
    return a


def _layer_rc(a):
    return _rc("mh_mamba2_layer_step_workspace_bytes", ct.byref(a), ct.byref(ct.c_size_t()))


def test_layer_step_refuses_overlapping_conv_states():
    a = _good_layer_step()
    assert _layer_rc(a) == 0
    a.conv_out = a.conv_state                           # the same rows in the same places
    assert _layer_rc(a) == 0
    span = 2 * 3 * 64 * 2
    for off in (2, -2, span - 2, 2 - span):
        a.conv_out = a.conv_state + off
        assert _layer_rc(a) == -4 and b"conv_out" in _lib.lib().mh_last_error(), off
    for off in (span, -span):
        a.conv_out = a.conv_state + off
        assert _layer_rc(a) == 0, off
    a = _good_layer_step(rows=2)                        # a row more comes out: rows move
    a.conv_out = a.conv_state
    assert _layer_rc(a) == -4
    a = _good_layer_step()                              # x's half of wider rows
    a.conv_state_stride_l, a.conv_state_stride_b = 128, 3 * 128
    a.conv_out = a.conv_state
    assert _layer_rc(a) == -4
    a.batch, a.conv_state_len, a.width = 1, 1, 2        # one row of one sequence: its strides say nothing
    assert _layer_rc(a) == 0
