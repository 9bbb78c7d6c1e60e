"""The kernels on state columns against the oracle, at the edges of their tiles: columns
shorter than a tile, of one tile and of several; one state (read in place, and copied when its
buffer is not 16-byte aligned), ragged last column groups, more than one slab; random and
structured string sets.

Bars, as for the other kernels: complex128 within 1e-12, complex64 (FP32 products, FP64 sums)
within 1e-5 of the FP64 oracle."""

import threading

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


def test_expectation_of_millions_of_strings(hip):
    """Strings and columns whose items at their usual size would make a launch of more than 2^32
    threads, of which HIP runs a part: larger items instead."""
    n, N, S = 9, 2_200_000, 16384
    H.say(f"expectation on columns n={n} N={N} S={S}")
    codes, coeffs = syn.random_codes(N, n, seed=1), syn.random_coeffs(N, seed=1)
    ops = _abi.Ops(codes, coeffs)
    assert _abi.op_expectation_columns(ops, C128, 1 << n, S)
    psi = syn.random_states(1 << n, S, seed=1)
    got = H.op_expectation(ops, psi, C128)[[0, S // 2, S - 1]]
    sample = np.ascontiguousarray(psi[:, [0, S // 2, S - 1]])
    assert H.ev_scaled_err(got, _oracle(codes, coeffs, sample), coeffs, sample) <= 1e-12


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


# ---------------------------------------------------------------------------
# apply: IEEE-equal to the oracle's sequential loop
# ---------------------------------------------------------------------------
def _odt(dtype):
    return O.C128 if dtype == C128 else O.C64


@pytest.mark.parametrize("dtype,n,S", [
    # one column made of the batch (power-of-two state counts), one wave to many
    (C128, 6, 1), (C128, 5, 2), (C128, 10, 16), (C128, 13, 1), (C64, 6, 1), (C64, 8, 4), (C64, 12, 128), (C64, 15, 1),
    # transposed columns: shorter and longer than a block, odd counts (complex64: a state paired with zeros)
    (C128, 6, 5), (C128, 7, 33), (C128, 9, 3), (C128, 13, 3), (C64, 6, 3), (C64, 7, 40), (C64, 10, 33), (C64, 14, 6),
    # tiles in LDS: columns shorter than a tile (a ragged last group), of one tile and of two
    (C128, 11, 771), (C128, 13, 193), (C128, 14, 97), (C64, 12, 771), (C64, 14, 195),
])
@pytest.mark.parametrize("kind", ["random", "weight2"])
def test_apply_on_columns(hip, monkeypatch, kind, dtype, n, S):
    H.say(f"apply on columns {kind} n={n} S={S} dtype={dtype}")
    monkeypatch.setenv("FAST_PAULI_APPLY_KERNEL", "columns")
    cdt = H.CDT[dtype]
    codes = _structured_codes(kind, 29, n, seed=n + S)
    strings = syn.codes_to_strings(codes)
    coeffs = syn.random_coeffs(29, seed=S + 2)
    ops = _abi.Ops(codes, coeffs)
    assert _abi.op_apply_columns(ops, dtype, 1 << n, S)
    psi = syn.random_states(1 << n, S, seed=n * 17 + S).astype(cdt)
    got = H.op_apply(ops, psi, dtype)
    assert np.array_equal(got, O.op_apply(strings, coeffs.astype(cdt), psi, np.zeros_like(psi), dtype=_odt(dtype)))
    base = syn.random_states(1 << n, S, seed=n + 12).astype(cdt)
    got = H.op_apply(ops, psi, dtype, out0=base)
    assert np.array_equal(got, O.op_apply(strings, coeffs.astype(cdt), psi, base.copy(), dtype=_odt(dtype)))


@pytest.mark.parametrize("N", [2, 3, 4, 5, 7, 8, 23, 24, 25, 48])
def test_apply_on_columns_string_counts(hip, monkeypatch, N):
    """Every remainder of the strings in flight and of the unrolled stages."""
    H.say(f"apply on columns N={N}")
    monkeypatch.setenv("FAST_PAULI_APPLY_KERNEL", "columns")
    for n, S in ((9, 4), (13, 200)):
        codes, coeffs = syn.random_codes(N, n, seed=N), syn.random_coeffs(N, seed=N)
        psi = syn.random_states(1 << n, S, seed=N + n)
        got = H.op_apply(_abi.Ops(codes, coeffs), psi, C128)
        assert np.array_equal(got, O.op_apply(syn.codes_to_strings(codes), coeffs, psi, np.zeros_like(psi)))


@pytest.mark.parametrize("dtype,n,N,K,S", [(C128, 8, 40, 3, 5), (C128, 14, 33, 9, 97), (C64, 9, 50, 7, 37),
                                           (C64, 14, 20, 4, 195), (C128, 12, 30, 5, 1), (C64, 11, 17, 300, 1)])
def test_summed_apply_on_columns(hip, monkeypatch, dtype, n, N, K, S):
    """SummedPauliOp::apply and apply_weighted (per-state weights), overwrite and accumulate."""
    H.say(f"summed apply on columns n={n} N={N} K={K} S={S} dtype={dtype}")
    monkeypatch.setenv("FAST_PAULI_APPLY_KERNEL", "columns")
    cdt = H.CDT[dtype]
    codes = syn.random_codes(N, n, seed=n * 5 + N)
    strings = syn.codes_to_strings(codes)
    rng = np.random.default_rng(n + N + K + S)
    coeffs_nk = rng.standard_normal((N, K)) + 1j * rng.standard_normal((N, K))
    ops = _abi.Ops(codes, matrix=coeffs_nk)
    psi = syn.random_states(1 << n, S, seed=n + S).astype(cdt)
    data = rng.standard_normal((K, S)).astype(np.float64 if dtype == C128 else np.float32)
    dim = 1 << n
    assert _abi.op_apply_columns(ops, dtype, dim, S) and _abi.op_apply_columns(ops, dtype, dim, S, weighted=True)
    d_in, d_data = _abi.DeviceBuffer.from_array(psi), _abi.DeviceBuffer.from_array(data)
    c_dt = coeffs_nk.astype(cdt)
    for base in (np.zeros_like(psi), syn.random_states(dim, S, seed=98).astype(cdt)):
        acc = int(base.any())
        d_out = _abi.DeviceBuffer.from_array(base)
        _abi.call("fp_hip_summed_apply", ops.handle, dtype, d_in.ptr, d_out.ptr, dim, S, acc, None)
        exp = O.summed_apply(strings, c_dt, psi, base.copy(), dtype=_odt(dtype))
        assert np.array_equal(d_out.to_array(cdt, psi.shape), exp)
        d_out.upload(base)
        _abi.call("fp_hip_summed_apply_weighted", ops.handle, dtype, d_in.ptr, d_data.ptr, d_out.ptr, dim, S, acc,
                  None)
        exp = O.summed_apply_weighted(strings, c_dt, psi, data, base.copy(), dtype=_odt(dtype))
        assert np.array_equal(d_out.to_array(cdt, psi.shape), exp)


def test_apply_on_columns_several_slabs_and_unaligned(hip, monkeypatch):
    """70 complex128 columns of 2 MiB (more than one 128 MiB slab), and complex64 buffers at 8
    bytes past a 16-byte boundary: equal to the streaming kernel, itself checked against the oracle."""
    H.say("apply on columns, several slabs and unaligned buffers")
    for dtype, n, S, off in ((C128, 17, 70, 0), (C64, 12, 64, 8), (C64, 12, 33, 8), (C64, 18, 3, 0)):
        cdt = H.CDT[dtype]
        ops = _abi.Ops(syn.random_codes(9, n, seed=n), syn.random_coeffs(9, seed=n))
        nbytes = (1 << n) * S * np.dtype(cdt).itemsize
        d_in, d_out = _abi.DeviceBuffer(nbytes + 16), _abi.DeviceBuffer(nbytes + 16)
        d_in.zero()
        d_in.upload(np.ascontiguousarray(syn.random_states(1 << n, S, seed=n).astype(cdt)))
        got = []
        for kernel in ("columns", "stream"):
            monkeypatch.setenv("FAST_PAULI_APPLY_KERNEL", kernel)
            d_out.zero()
            # the last state's end is outside the uploaded array when shifted: still inside the buffer
            _abi.call("fp_hip_op_apply", ops.handle, dtype, d_in.ptr + off, d_out.ptr + off, 1 << n, S, 0, None)
            got.append(d_out.to_array(np.uint8, (nbytes + 16,)).copy())
        assert np.array_equal(got[0], got[1]), (dtype, n, S, off)


def test_apply_columns_rule(hip, monkeypatch):
    """Which shapes run on columns; the rest, and the other kernels when forced, do not."""
    H.say("apply columns rule")
    for n, N, S, want in ((10, 64, 128, True), (18, 1000, 1, True), (14, 500, 1000, True), (12, 64, 100, False),
                          (20, 24, 1, False), (21, 96, 8, False), (10, 1, 128, False)):
        ops = _abi.Ops(syn.random_codes(N, n, seed=n))
        assert _abi.op_apply_columns(ops, C128, 1 << n, S) == want, (n, N, S)
    # one complex64 state past 2 MiB, and weights of one state, pay from more strings on
    for n, N, want in ((18, 2, True), (19, 15, False), (19, 16, True), (20, 63, False), (20, 64, True)):
        ops = _abi.Ops(syn.random_codes(N, n, seed=n))
        assert _abi.op_apply_columns(ops, C64, 1 << n, 1) == want, (n, N)
    for N, want in ((7, False), (8, True)):
        assert _abi.op_apply_columns(_abi.Ops(syn.random_codes(N, 10, seed=N)), C128, 1 << 10, 1, weighted=True) == want
    # weights per state: from 48 strings on small batches too
    for n, N, S, want in ((10, 48, 2, True), (10, 47, 2, False), (18, 48, 2, False), (18, 48, 3, True)):
        ops = _abi.Ops(syn.random_codes(N, n, seed=n))
        assert _abi.op_apply_columns(ops, C128, 1 << n, S, weighted=True) == want, (n, N, S)
    monkeypatch.setenv("FAST_PAULI_APPLY_KERNEL", "tiled")
    assert not _abi.op_apply_columns(_abi.Ops(syn.random_codes(64, 10, seed=1)), C128, 1 << 10, 128)


@pytest.mark.parametrize("dtype,n,S", [(C128, 12, 9), (C64, 15, 1), (C64, 13, 6)])
def test_columns_follow_assign_and_coeffs(hip, monkeypatch, dtype, n, S):
    """Re-targeted sets (more strings, fewer, others) and new coefficients: the expectation's cached
    items and the apply's masks and coefficients are those of a fresh set."""
    H.say(f"columns after assign / set_coeffs n={n} S={S} dtype={dtype}")
    monkeypatch.setenv("FAST_PAULI_EV_KERNEL", "columns")
    monkeypatch.setenv("FAST_PAULI_APPLY_KERNEL", "columns")
    psi = syn.random_states(1 << n, S, seed=31).astype(H.CDT[dtype])
    ops = _abi.Ops(syn.random_codes(64, n, seed=31), syn.random_coeffs(64, seed=31))

    def same_as(fresh):
        assert _abi.op_expectation_columns(ops, dtype, 1 << n, S) and _abi.op_apply_columns(ops, dtype, 1 << n, S)
        assert np.array_equal(H.op_expectation(ops, psi, dtype), H.op_expectation(fresh, psi, dtype))
        assert np.array_equal(H.op_apply(ops, psi, dtype), H.op_apply(fresh, psi, dtype))

    same_as(_abi.Ops(syn.random_codes(64, n, seed=31), syn.random_coeffs(64, seed=31)))
    for N, seed in ((300, 32), (40, 33), (300, 34)):
        codes, coeffs = syn.random_codes(N, n, seed=seed), syn.random_coeffs(N, seed=seed)
        ops.assign(codes, coeffs)
        _abi.synchronize()
        same_as(_abi.Ops(codes, coeffs))
    coeffs = syn.random_coeffs(300, seed=35)
    ops.set_coeffs(coeffs)
    same_as(_abi.Ops(codes, coeffs))
    want = _oracle(codes, coeffs, psi)
    assert H.ev_scaled_err(H.op_expectation(ops, psi, dtype), want, coeffs, psi) <= (1e-12 if dtype == C128 else 1e-5)


# ---------------------------------------------------------------------------
# streams, threads and captured graphs
# ---------------------------------------------------------------------------
PER_THREAD = 2  # the handle hipStreamPerThread: another stream in every host thread


def test_columns_on_per_thread_streams(hip):
    """One handle, two host threads, two streams: the transposed slabs (and partials) are each
    thread's own.  Applies IEEE-equal, expectation values identical, to the null stream's."""
    H.say("columns on per-thread streams")
    n, N, S, rounds = 15, 64, 45, 12  # 23 MB of columns: the threads' kernels overlap
    work = []
    for seed in (1, 2):
        ops = _abi.Ops(syn.random_codes(N, n, seed=seed), syn.random_coeffs(N, seed=seed))
        assert _abi.op_apply_columns(ops, C128, 1 << n, S)
        psi = syn.random_states(1 << n, S, seed=seed)
        want = H.op_apply(ops, psi, C128), H.op_expectation(ops, psi, C128)
        outs = [_abi.DeviceBuffer(psi.nbytes) for _ in range(rounds)]
        evs = [_abi.DeviceBuffer(S * 16) for _ in range(rounds)]
        work.append((ops, _abi.DeviceBuffer.from_array(psi), outs, evs, want, psi.shape))
    _abi.synchronize()
    failed, go = [], threading.Barrier(2)

    def body(ops, d_in, outs, evs, *_):
        try:
            go.wait(timeout=30)
            for d_out, d_ev in zip(outs, evs):
                _abi.call("fp_hip_op_apply", ops.handle, C128, d_in.ptr, d_out.ptr, 1 << n, S, 0, PER_THREAD)
                _abi.call("fp_hip_op_expectation", ops.handle, C128, d_in.ptr, d_ev.ptr, 1 << n, S, 0, PER_THREAD)
            _abi.call("fp_hip_stream_synchronize", PER_THREAD)
        except Exception as e:  # reported by the main thread
            failed.append(e)

    threads = [threading.Thread(target=body, args=w) for w in work]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
    for _, _, outs, evs, (apply, ev), shape in work:
        for d_out, d_ev in zip(outs, evs):
            assert np.array_equal(d_out.to_array(np.complex128, shape), apply)
            assert np.array_equal(d_ev.to_array(np.complex128, (S,)), ev)


def test_captured_scratch_outlives_larger_calls(hip, monkeypatch):
    """A graph holds the scratch its stream had at the capture: an apply on columns, which needs
    more, takes another buffer.  Replays, with eager work between them, equal the eager call."""
    H.say("captured expectation beside larger applies")
    stream = _abi.Stream()
    n, N, S = 10, 12, 5
    ops = _abi.Ops(syn.random_codes(N, n, seed=3), syn.random_coeffs(N, seed=3))
    psi = syn.random_states(1 << n, S, seed=3)
    d_in, d_out = _abi.DeviceBuffer.from_array(psi), _abi.DeviceBuffer(S * 16)

    def expect(handle):
        _abi.call("fp_hip_op_expectation", ops.handle, C128, d_in.ptr, d_out.ptr, 1 << n, S, 0, handle)

    monkeypatch.setenv("FAST_PAULI_EV_KERNEL", "stream")
    expect(stream.handle)
    stream.synchronize()
    want = d_out.to_array(np.complex128, (S,))
    graph = H.Graph(stream, expect)
    for m, T in ((13, 70), (14, 90), (15, 100)):  # scratch of 18, 47 and 105 MB
        big = _abi.Ops(syn.random_codes(64, m, seed=m), syn.random_coeffs(64, seed=m))
        phi = syn.random_states(1 << m, T, seed=m)
        d_phi, d_big = _abi.DeviceBuffer.from_array(phi), _abi.DeviceBuffer(phi.nbytes)
        assert _abi.op_apply_columns(big, C128, 1 << m, T)
        _abi.call("fp_hip_op_apply", big.handle, C128, d_phi.ptr, d_big.ptr, 1 << m, T, 0, stream.handle)
        d_out.zero()
        _abi.synchronize()
        graph.replay()
        assert np.array_equal(d_out.to_array(np.complex128, (S,)), want)
        assert np.array_equal(d_big.to_array(np.complex128, phi.shape), H.op_apply(big, phi, C128))
    graph.destroy()
    stream.destroy()


@pytest.mark.parametrize("mode", [0, 2], ids=["global", "relaxed"])
@pytest.mark.parametrize("warm", [True, False], ids=["warm", "cold"])
@pytest.mark.parametrize("entry,dtype,n,N,S", [
    ("fp_hip_op_expectation", C128, 14, 64, 40),   # columns
    ("fp_hip_op_expectation", C64, 15, 70, 1),     # one state, read in place
    ("fp_hip_op_expectation", C128, 14, 16, 16),   # coset-tiled
    ("fp_hip_op_expectation", C128, 9, 1, 3),      # streaming
    ("fp_hip_op_expectation_noalloc", C128, 14, 64, 40),
    ("fp_hip_op_apply", C128, 10, 40, 16),         # one column made of the batch
    ("fp_hip_op_apply", C64, 14, 100, 80),         # transposed columns: streaming in the graph
    ("fp_hip_op_apply", C128, 14, 100, 300),       # transposed columns: coset-tiled in the graph
    ("fp_hip_summed_apply_weighted", C128, 10, 50, 3),
])
def test_captured_calls(hip, entry, dtype, n, N, S, warm, mode):
    """Captured on the stream that an eager call warmed, or without one: every replay, with eager
    work on the set between them, gives the eager call's bits."""
    H.say(f"captured {entry} n={n} N={N} S={S} dtype={dtype} warm={warm} mode={mode}")
    K, cdt = 4, H.CDT[dtype]
    codes = syn.random_codes(N, n, seed=n + N)
    rng = np.random.default_rng(N)
    weighted = entry == "fp_hip_summed_apply_weighted"
    make = (lambda: _abi.Ops(codes, matrix=mat)) if weighted else (lambda: _abi.Ops(codes, coeffs))
    mat, coeffs = rng.standard_normal((N, K)) + 0j, syn.random_coeffs(N, seed=N)
    psi = syn.random_states(1 << n, S, seed=N).astype(cdt)
    shape = (S,) if "expectation" in entry else psi.shape
    d_in = _abi.DeviceBuffer.from_array(psi)
    data = rng.standard_normal((K, S)).astype(np.float64 if dtype == C128 else np.float32)
    d_data = _abi.DeviceBuffer.from_array(data)
    d_out = _abi.DeviceBuffer(int(np.prod(shape)) * np.dtype(cdt).itemsize)
    args = [d_in.ptr] + ([d_data.ptr] if weighted else []) + [d_out.ptr, 1 << n, S, 0]

    def run(ops, handle):
        _abi.call(entry, ops.handle, dtype, *args, handle)

    run(make(), None)  # another set, on another stream
    _abi.synchronize()
    want = d_out.to_array(cdt, shape)
    ops, stream = make(), _abi.Stream()
    if warm:
        run(ops, stream.handle)
        stream.synchronize()
    graph = H.Graph(stream, lambda handle: run(ops, handle), mode)
    for rep in range(3):
        d_out.zero()
        _abi.synchronize()
        graph.replay()
        assert np.array_equal(d_out.to_array(cdt, shape), want), rep
        run(ops, stream.handle if rep else None)
        _abi.synchronize()
        assert np.array_equal(d_out.to_array(cdt, shape), want), rep
    graph.destroy()
    stream.destroy()
