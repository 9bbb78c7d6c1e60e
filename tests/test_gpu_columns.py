"""The kernels on state columns against the oracle, at the edges of their tiles: columns
shorter than a tile, of one tile and of several; one state (read in place, and copied when its
buffer is not 16-byte aligned), ragged last column groups, more than one slab; random and
structured string sets.

Bars, as for the other kernels: complex128 within 1e-12, complex64 (FP32 products, FP64 sums)
within 1e-5 of the FP64 oracle."""

import numpy as np
import pytest

from fast_pauli import _abi
from fast_pauli import synthetic as syn
from oracle import oracle as O
from tests import hiputil as H
from tests.test_gpu_hotpath import _structured_codes

pytestmark = pytest.mark.gpu

C128, C64 = _abi.FP_C128, _abi.FP_C64


def _oracle(codes, coeffs, psi):
    return O.op_expectation(syn.codes_to_strings(codes), coeffs, psi.astype(np.complex128),
                            np.zeros(psi.shape[1], np.complex128), par=True)


@pytest.mark.parametrize("dtype,n,S", [
    (C128, 9, 1), (C128, 9, 13), (C128, 10, 40), (C128, 11, 2), (C128, 12, 5), (C128, 13, 1), (C128, 14, 33),
    (C128, 15, 3), (C64, 10, 1), (C64, 10, 21), (C64, 11, 40), (C64, 12, 3), (C64, 13, 1), (C64, 13, 34),
    (C64, 14, 7), (C64, 16, 2),
])
@pytest.mark.parametrize("kind", ["random", "weight2", "diagonal", "shared_x", "duplicates"])
def test_expectation_on_columns(hip, monkeypatch, kind, dtype, n, S):
    H.say(f"expectation on columns {kind} n={n} S={S} dtype={dtype}")
    monkeypatch.setenv("FAST_PAULI_EV_KERNEL", "columns")
    codes = _structured_codes(kind, 70, n, seed=n + S)
    coeffs = syn.random_coeffs(codes.shape[0], seed=S + 1)
    ops = _abi.Ops(codes, coeffs)
    assert _abi.op_expectation_columns(ops, dtype, 1 << n, S)
    psi = syn.random_states(1 << n, S, seed=n * 31 + S).astype(H.CDT[dtype])
    got = H.op_expectation(ops, psi, dtype)
    exp = _oracle(codes, coeffs, psi)
    tol = 1e-12 if dtype == C128 else 1e-5
    assert H.ev_scaled_err(got, exp, coeffs, psi) <= tol
    assert np.array_equal(H.op_expectation(ops, psi, dtype), got)
    base = syn.random_coeffs(S, seed=3).astype(H.CDT[dtype])
    assert H.rel_err(H.op_expectation(ops, psi, dtype, out0=base) - base, exp) <= 10 * tol


def test_expectation_on_columns_several_slabs(hip, monkeypatch):
    """150 columns of 1 MiB: more than one 128 MiB slab."""
    H.say("expectation on columns, several slabs")
    monkeypatch.setenv("FAST_PAULI_EV_KERNEL", "columns")
    n, N, S = 16, 8, 150
    codes, coeffs = syn.random_codes(N, n, seed=5), syn.random_coeffs(N, seed=5)
    psi = syn.random_states(1 << n, S, seed=6)
    got = H.op_expectation(_abi.Ops(codes, coeffs), psi, C128)
    assert H.ev_scaled_err(got, _oracle(codes, coeffs, psi), coeffs, psi) <= 1e-12


def test_expectation_on_columns_unaligned_state(hip, monkeypatch):
    """One complex64 state at 8 bytes past a 16-byte boundary (the ABI asks for 8): copied."""
    H.say("expectation on columns, unaligned state")
    monkeypatch.setenv("FAST_PAULI_EV_KERNEL", "columns")
    n, N = 14, 30
    codes, coeffs = syn.random_codes(N, n, seed=7), syn.random_coeffs(N, seed=7)
    ops = _abi.Ops(codes, coeffs)
    psi = syn.random_states(1 << n, 1, seed=8).astype(np.complex64)
    d_in = _abi.DeviceBuffer.from_array(np.concatenate([np.zeros((1, 1), np.complex64), psi]))
    d_out = _abi.DeviceBuffer(8)
    _abi.call("fp_hip_op_expectation", ops.handle, C64, d_in.ptr + 8, d_out.ptr, 1 << n, 1, 0, None)
    got = d_out.to_array(np.complex64, (1,))
    assert H.ev_scaled_err(got, _oracle(codes, coeffs, psi), coeffs, psi) <= 1e-5
    assert np.array_equal(got, H.op_expectation(ops, psi, C64))


def test_expectation_columns_rule(hip, monkeypatch):
    """Full classes take columns, a few strings on many tiles do not; the sizes a tile cannot
    take never do; the other kernels can be forced."""
    H.say("expectation columns rule")
    for n, N, S, want in ((14, 1024, 100, True), (16, 1024, 1, True), (14, 16, 16, False), (20, 128, 16, False),
                          (8, 500, 4, False), (24, 256, 16, False)):
        ops = _abi.Ops(syn.random_codes(N, n, seed=n))
        assert _abi.op_expectation_columns(ops, C128, 1 << n, S) == want, (n, N, S)
    monkeypatch.setenv("FAST_PAULI_EV_KERNEL", "tiled")
    ops = _abi.Ops(syn.random_codes(1024, 14, seed=1))
    assert not _abi.op_expectation_columns(ops, C128, 1 << 14, 100)
    with pytest.raises(ValueError):
        _abi.op_expectation_columns(ops, C128, 1 << 13, 100)
