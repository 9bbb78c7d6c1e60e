"""The workloads whose speed is measured, one pass each through the public entry points.

A case is a dict of plain values.  `listed()` names the fixed cases, `draw(rng)` makes
another one of the same ranges, `prepare(case, seed)` makes what a program holds before
the call (device-resident states and operator sets), `run(state)` is one pass,
`exact(case, seed)` the same result in 64 bits from plain torch, and `work(case)` the bytes
and operations a pass cannot do without.

Device-resident work goes through the C ABI (`fast_pauli._abi`, the binding the tests and
the benchmark use) with torch tensors as device memory; the host-array case goes through the
Python module, whose calls take and return numpy arrays.
"""

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fast-pauli_amd"))


def listed():
    return [
        # the smallest calls: a small operator on a batch that lives in the caches (launch bound)
        {"name": "apply_n10_s128_c128", "kind": "op_apply", "n": 10, "strings": 64, "states": 128, "c64": False},
        # one state vector and a long operator: the step of a time evolution or a Krylov solver
        {"name": "apply_n18_s1_c128", "kind": "op_apply", "n": 18, "strings": 1000, "states": 1, "c64": False},
        # a large serving request with a ragged state count, in the fast precision
        {"name": "apply_n20_s19_c64", "kind": "op_apply", "n": 20, "strings": 512, "states": 19, "c64": True},
        # one string on the largest batch: pure memory traffic
        {"name": "string_n24_s16_c128", "kind": "string_apply", "n": 24, "strings": 1, "states": 16, "c64": False},
        # the energy of one state under a long Hamiltonian: the inner loop of a variational solver
        {"name": "ev_n16_s1_c128", "kind": "op_ev", "n": 16, "strings": 1024, "states": 1, "c64": False},
        # the same over a data set of states
        {"name": "ev_n14_s1000_c128", "kind": "op_ev", "n": 14, "strings": 1024, "states": 1000, "c64": False},
        # a serving request: medium, ragged, fast precision
        {"name": "ev_n18_s13_c64", "kind": "op_ev", "n": 18, "strings": 300, "states": 13, "c64": True},
        # the largest expectation value, beyond every cache
        {"name": "ev_n24_s16_c128", "kind": "op_ev", "n": 24, "strings": 256, "states": 16, "c64": False},
        # expectation values through the Python module, numpy in and numpy out (copies included)
        {"name": "py_ev_n12_s100_c128", "kind": "py_ev", "n": 12, "strings": 1024, "states": 100, "c64": False},
        # many observables over a data set of states ...
        {"name": "summed_ev_n14_c128", "kind": "summed_ev", "n": 14, "strings": 2000, "operators": 200,
         "states": 1000, "c64": False, "contraction": 3},
        # ... and their weighted sum applied to each state, with weights of its own
        {"name": "summed_weighted_n14_c128", "kind": "summed_weighted", "n": 14, "strings": 2000, "operators": 200,
         "states": 1000, "c64": False},
        # many operators of uneven size in one graph launch
        {"name": "batch_256_c64", "kind": "batch", "operators": 256, "c64": True},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["op_apply", "op_apply", "op_apply", "string_apply", "op_ev", "op_ev", "op_ev", "py_ev",
                       "summed_ev", "summed_weighted", "summed_apply", "batch"])
    c64 = rng.random() < 0.4
    if kind == "batch":
        return {"kind": kind, "operators": _log_int(rng, 16, 240), "c64": True}
    if kind == "string_apply":
        n = rng.randint(8, 24)
        return {"kind": kind, "n": n, "strings": 1, "states": _log_int(rng, 1, min(128, 1 << (28 - n))), "c64": c64}
    if kind in ("op_apply", "op_ev"):
        n = rng.randint(8, 22 if kind == "op_apply" else 24)
        states = _log_int(rng, 1, min(128 if kind == "op_apply" else 1000, 1 << (28 - n)))
        room = (1e10 if kind == "op_apply" else 6.5e10) / ((1 << n) * states)
        return {"kind": kind, "n": n, "strings": _log_int(rng, 8, int(max(8, min(1024, room)))), "states": states,
                "c64": c64}
    n = rng.randint(8, 14)
    states = _log_int(rng, 1, 1000)
    case = {"kind": kind, "n": n, "strings": _log_int(rng, 16, 1024 if kind == "py_ev" else 2000), "states": states,
            "c64": c64}
    if kind != "py_ev":
        case["operators"] = _log_int(rng, 2, 200)
    if kind == "summed_ev":
        case["contraction"] = rng.choice([2, 3, 3]) if c64 else 3
    return case


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------

def _codes(r, n_strings, n):
    """Letter codes 0..3 = I, X, Y, Z, every site uniform."""
    return r.integers(0, 4, size=(n_strings, n), dtype=np.uint8)


def _codes_weight3(r, n_strings, n):
    """Strings of weight 1..3: support sites uniform, letters uniform over X, Y, Z."""
    out = np.zeros((n_strings, n), np.uint8)
    weight = r.integers(1, 4, size=n_strings)
    sites = np.argsort(r.random((n_strings, n)), axis=1)
    letters = r.integers(1, 4, size=(n_strings, 3), dtype=np.uint8)
    rows = np.arange(n_strings)
    for k in range(3):
        live = k < np.minimum(weight, n)
        out[rows[live], sites[live, k]] = letters[live, k]
    return out


def _coeffs(r, count):
    return r.standard_normal(count) + 1j * r.standard_normal(count)


def _states(seed, dim, n_states, c64):
    """Normalised random states on the GPU, (dim, n_states) row-major."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    re = torch.float32 if c64 else torch.float64
    psi = torch.view_as_complex(torch.randn(dim, n_states, 2, generator=g, device="cuda", dtype=re))
    return psi.div_(torch.linalg.vector_norm(psi, dim=0, keepdim=True))


def _batch_shapes(case, r):
    """Sizes of an uneven batch: n uniform in 8..18, 16..512 strings, 1..64 states."""
    shapes = []
    for _ in range(case["operators"]):
        n = int(r.integers(8, 19))
        strings = int(round(math.exp(r.uniform(math.log(16), math.log(512)))))
        shapes.append((n, strings, int(r.integers(1, 65))))
    return shapes


def _batch_inputs(case, seed):
    r = np.random.default_rng(seed)
    # the sizes belong to the case, so that every seed is the same amount of work
    shapes = _batch_shapes(case, np.random.default_rng(case["operators"]))
    ops, total = [], 0
    for n, strings, states in shapes:
        # entries start at multiples of 64 elements, as allocations of their own would be aligned
        ops.append({"n": n, "states": states, "codes": _codes(r, strings, n), "coeffs": _coeffs(r, strings),
                    "at": total})
        total += -(-((1 << n) * states) // 64) * 64
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    psi = torch.view_as_complex(torch.randn(total, 2, generator=g, device="cuda", dtype=torch.float32))
    for e in ops:
        dim = 1 << e["n"]
        block = psi[e["at"]:e["at"] + dim * e["states"]].view(dim, e["states"])
        block.div_(torch.linalg.vector_norm(block, dim=0, keepdim=True))
    return ops, psi


def _inputs(case, seed):
    r = np.random.default_rng(seed)
    kind, n, strings = case["kind"], case["n"], case["strings"]
    summed = kind.startswith("summed")
    got = {"codes": _codes_weight3(r, strings, n) if summed else _codes(r, strings, n),
           "coeffs": _coeffs(r, strings)}
    if summed:
        got["matrix"] = r.standard_normal((strings, case["operators"]))
    if kind == "summed_weighted":
        got["data"] = r.standard_normal((case["operators"], case["states"]))
        if case["c64"]:
            got["data"] = got["data"].astype(np.float32)
    got["states"] = _states(seed, 1 << n, case["states"], case["c64"])
    return got


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def prepare(case, seed):
    from fast_pauli import _abi

    _abi.init(0)
    dtype = _abi.FP_C64 if case["c64"] else _abi.FP_C128
    state = {"kind": case["kind"], "dtype": dtype}
    if case["kind"] == "batch":
        from fast_pauli.batch import Batch

        entries, psi = _batch_inputs(case, seed)
        out = torch.zeros_like(psi)
        batch = Batch()
        for e in entries:
            at = e["at"] * psi.element_size()
            batch.add_apply(_abi.Ops(e["codes"], e["coeffs"]), psi.data_ptr() + at, out.data_ptr() + at,
                            1 << e["n"], e["states"], dtype)
        return dict(state, batch=batch, states=psi, out=out)
    got = _inputs(case, seed)
    psi = got["states"]
    dim, n_states = psi.shape
    state.update(states=psi, dim=dim, n_states=n_states)
    if case["kind"] == "py_ev":
        import fast_pauli as fp

        strings = ["".join("IXYZ"[c] for c in row) for row in got["codes"]]
        return {"kind": "py_ev", "op": fp.PauliOp(list(got["coeffs"]), strings), "states": psi.cpu().numpy()}
    state["ops"] = _abi.Ops(got["codes"], got["coeffs"], matrix=got.get("matrix"))
    if case["kind"] == "op_ev":
        state["out"] = torch.zeros(n_states, dtype=psi.dtype, device="cuda")
    elif case["kind"] == "summed_ev":
        state["out"] = torch.zeros(case["operators"], n_states, dtype=psi.dtype, device="cuda")
        state["contraction"] = case["contraction"]
    else:
        state["out"] = torch.zeros_like(psi)
    if case["kind"] == "summed_weighted":
        state["data"] = torch.from_numpy(got["data"]).cuda()
    return state


def run(state):
    from fast_pauli import _abi

    kind = state["kind"]
    if kind == "py_ev":
        return state["op"].expectation_value(state["states"])
    out = state["out"]
    if kind == "batch":
        state["batch"].launch()
        return out
    ops, dtype, dim, n_states = state["ops"].handle, state["dtype"], state["dim"], state["n_states"]
    p_in, p_out = state["states"].data_ptr(), out.data_ptr()
    if kind == "string_apply":
        _abi.call("fp_hip_string_apply_batch", ops, 0, dtype, p_in, p_out, dim, n_states, 1.0, 0.0, 0, None)
    elif kind == "op_apply":
        _abi.call("fp_hip_op_apply", ops, dtype, p_in, p_out, dim, n_states, 0, None)
    elif kind == "op_ev":
        _abi.call("fp_hip_op_expectation", ops, dtype, p_in, p_out, dim, n_states, 0, None)
    elif kind == "summed_ev":
        _abi.call("fp_hip_summed_expectation", ops, dtype, state["contraction"], p_in, p_out, dim, n_states, 0, None)
    elif kind == "summed_apply":
        _abi.call("fp_hip_summed_apply", ops, dtype, p_in, p_out, dim, n_states, 0, None)
    else:
        _abi.call("fp_hip_summed_apply_weighted", ops, dtype, p_in, state["data"].data_ptr(), p_out, dim, n_states,
                  0, None)
    return out


# ---------------------------------------------------------------------------
# the same results in 64 bits, from plain torch
# ---------------------------------------------------------------------------

class _Dense:
    """P psi for one string at a time: (P psi)_j = (-i)^{nY} (-1)^{popcount(j & z)} psi_{j ^ x}."""

    def __init__(self, n):
        self.n = n
        self.j = torch.arange(1 << n, device="cuda", dtype=torch.int64)
        par = self.j.clone()
        for s in (16, 8, 4, 2, 1):
            par ^= par >> s
        self.sign = 1.0 - 2.0 * (par & 1).double()  # (-1)^{popcount(j)}

    def term(self, codes):
        """(partner rows, row values) of one string."""
        x = z = n_y = 0
        for i, c in enumerate(codes.tolist()):
            bit = 1 << (self.n - 1 - i)
            x |= bit if c in (1, 2) else 0
            z |= bit if c in (2, 3) else 0
            n_y += c == 2
        return self.j ^ x, (1, -1j, -1, 1j)[n_y % 4], self.sign[self.j & z]


def _exact_apply(n, codes, weights, psi):
    """sum_s weights[s] P_s psi; weights[s] a number or one number per state."""
    dense, out = _Dense(n), torch.zeros_like(psi)
    for s in range(len(codes)):
        partner, phase, sign = dense.term(codes[s])
        out.add_((psi[partner] * sign[:, None]) * (weights[s] * phase))
    return out


def _exact_ev(n, codes, psi):
    """(strings, states): <psi_t| P_s |psi_t>."""
    dense = _Dense(n)
    ev = torch.zeros(len(codes), psi.shape[1], dtype=torch.float64, device="cuda")
    conj = psi.conj()
    for s in range(len(codes)):
        partner, phase, sign = dense.term(codes[s])
        w = psi[partner].mul_(conj)
        ev[s] = ((sign @ w.real if phase in (1, -1) else sign @ w.imag)
                 * {1: 1.0, -1: -1.0, -1j: 1.0, 1j: -1.0}[phase])
        del w
    return ev


def _kept(coeffs, c64):
    """The coefficients as the entry points hold them."""
    c = np.asarray(coeffs)
    return c.astype(np.complex64).astype(np.complex128) if c64 else c.astype(np.complex128)


def exact(case, seed):
    kind, c64 = case["kind"], case["c64"]
    if kind == "batch":
        entries, psi = _batch_inputs(case, seed)
        out = torch.zeros(psi.shape, dtype=torch.complex128, device="cuda")
        for e in entries:
            dim, states = 1 << e["n"], e["states"]
            block = psi[e["at"]:e["at"] + dim * states].view(dim, states).to(torch.complex128)
            got = _exact_apply(e["n"], e["codes"], _kept(e["coeffs"], c64).tolist(), block)
            out[e["at"]:e["at"] + dim * states] = got.reshape(-1)
        return out
    got = _inputs(case, seed)
    n, codes, psi = case["n"], got["codes"], got["states"].to(torch.complex128)
    if kind == "string_apply":
        return _exact_apply(n, codes, [1.0], psi)
    if kind == "op_apply":
        return _exact_apply(n, codes, _kept(got["coeffs"], c64).tolist(), psi)
    if kind in ("op_ev", "py_ev"):
        c = torch.from_numpy(got["coeffs"]).cuda()
        value = (c[:, None] * _exact_ev(n, codes, psi)).sum(dim=0)
        return value.cpu().numpy() if kind == "py_ev" else value
    h = torch.from_numpy(got["matrix"]).cuda()
    if kind == "summed_ev":
        return torch.mm(h.T.contiguous(), _exact_ev(n, codes, psi)).to(torch.complex128)
    if c64:
        h = h.float().double()
    if kind == "summed_apply":
        return _exact_apply(n, codes, h.sum(dim=1).tolist(), psi)
    return _exact_apply(n, codes, torch.mm(h, torch.from_numpy(got["data"]).cuda().double()), psi)


def work(case):
    """Every state read once, every output written once; per (string, row, state) of an apply one
    complex product and one complex sum, of an expectation value half a pair's real product."""
    size = 8 if case["c64"] else 16
    if case["kind"] == "batch":
        shapes = _batch_shapes(case, np.random.default_rng(case["operators"]))
        return {"bytes": sum(2 * size * (1 << n) * t for n, _, t in shapes),
                "flops": sum(8 * s * (1 << n) * t for n, s, t in shapes)}
    elements = (1 << case["n"]) * case["states"]
    if case["kind"] in ("op_ev", "py_ev"):
        return {"bytes": size * (elements + case["states"]), "flops": 2 * case["strings"] * elements}
    if case["kind"] == "summed_ev":
        k = case["operators"]
        return {"bytes": size * (elements + k * case["states"]) + 8 * case["strings"] * k,
                "flops": 2 * case["strings"] * (elements + k * case["states"])}
    if case["kind"] == "string_apply":
        return {"bytes": 2 * size * elements, "flops": 6 * elements}
    flops, extra = 8 * case["strings"] * elements, 0
    if case["kind"] == "summed_weighted":
        flops += 2 * case["strings"] * case["operators"] * case["states"]
        extra = size // 2 * case["operators"] * (case["strings"] + case["states"])
    return {"bytes": 2 * size * elements + extra, "flops": flops}
