"""The workloads this library's speed is judged by: the calls a program that
uses it makes, over the sizes it makes them with.

Every case is a plain dict with a "kind":

  pair     one pairwise contraction of small host tensors (one step of a
           small tensor network): call latency
  theta    the two-site tensor of a large MPS as one pairwise contraction of
           device-resident tensors, written in another leg order
  net      contract(net) of the QFT expectation network in ncon's default
           order or the treewidth order
  svd      contract_svd of two host tensors (two truncated SVDs and the
           product of what they keep)
  circuit  a brick-wall circuit on a device MPS: per gate or per layer,
           complex FP64 or the chosen form, Haar or weakly entangling gates
  batch    many independent circuits advanced together
  expect   <psi|H|psi> of the transverse-field Ising chain, FP64 or BF16x3
  zipup    H|psi> compressed by zip-up
  mlp      training of the rank predictor (FP32)

listed() names twelve of them, draw(rng) makes more of the same ranges.  The
states of two implementations agree up to the gauge of their bonds, so an
MPS is returned by what no gauge changes: every bond spectrum, all (up to
2^12) or 256 amplitudes, <Z> of every site, the kept ranks and each update's
kept weight.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "qaintensor.jl_amd"))

from qaintensor import (DeviceMPO, DeviceMPS, FORM_CHOSEN,  # noqa: E402
                        FORM_PLAIN, _lib as L, circuits as C, contract,
                        contract_rep, default_context, hamiltonians as H,
                        learned, ops, run_circuits, workloads as W)
from qaintensor import network2graph as NG  # noqa: E402

FORMS = {"plain": FORM_PLAIN, "chosen": FORM_CHOSEN}


def listed():
    return [
        # a single step of a small network (the reference's test sizes):
        # latency of one call with host tensors, ragged legs
        dict(name="pair-small", kind="pair", a=13, b=2, c=17, d=19),
        # theta of two sites at chi = 500 (ragged), device to device
        dict(name="theta-500", kind="theta", l=500, m=511, r=489,
             order="2143"),
        # contract() of the 20-qubit QFT network after
        # optimize_contraction_order!: hundreds of tiny steps
        dict(name="net-qft20-treewidth", kind="net", n=20,
             order="treewidth"),
        # contract() without planning: the intermediates grow
        dict(name="net-qft17-default", kind="net", n=17, order="default"),
        # contract_svd of host tensors, ragged, truncating
        dict(name="svd-contract", kind="svd", a=30, b=21, c=100, d=25, e=22,
             er=1e-3),
        # a small circuit, one gate at a time, every amplitude wanted
        dict(name="circuit-12q-pergate", kind="circuit", n=12, depth=8,
             chi=32, cutoff=1e-10, form="plain", batched=False,
             gates="haar"),
        # the headline circuit in complex FP64, a layer per call
        dict(name="circuit-40q-fp64", kind="circuit", n=40, depth=20,
             chi=256, cutoff=1e-8, form="plain", batched=True, gates="haar"),
        # the headline circuit in the chosen form
        dict(name="circuit-40q-chosen", kind="circuit", n=40, depth=20,
             chi=256, cutoff=1e-8, form="chosen", batched=True,
             gates="haar"),
        # many uneven circuits at once, FP64
        dict(name="batch-24", kind="batch", count=24, chi=128, cutoff=1e-8,
             form="plain"),
        # <H> of a chi = 1024 random MPS in BF16x3
        dict(name="expect-1024-bf16x3", kind="expect", n=24, chi=1024,
             form="chosen"),
        # H|psi> by zip-up, recompressed to the same bond
        dict(name="zipup-128", kind="zipup", n=24, chi=128, cutoff=1e-10),
        # the rank predictor's training: 128 Adam steps on minibatches
        dict(name="mlp-train", kind="mlp", nb=4096, minibatch=256,
             steps=128),
    ]


def _log(rng, lo, hi):
    """An integer spread over [lo, hi] by its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pair", "theta", "net", "svd", "circuit", "circuit",
                       "circuit", "batch", "expect", "zipup", "mlp"])
    if kind == "pair":
        return dict(kind=kind, a=_log(rng, 3, 40), b=rng.randint(1, 5),
                    c=_log(rng, 2, 40), d=_log(rng, 3, 40))
    if kind == "theta":
        return dict(kind=kind, l=_log(rng, 40, 500), m=_log(rng, 40, 511),
                    r=_log(rng, 40, 489),
                    order=rng.choice(["1234", "2143", "1324", "4321"]))
    if kind == "net":
        order = rng.choice(["treewidth", "default"])
        return dict(kind=kind, n=rng.randint(6, 20 if order == "treewidth"
                                             else 17), order=order)
    if kind == "svd":
        return dict(kind=kind, a=rng.randint(3, 30), b=rng.randint(3, 21),
                    c=_log(rng, 8, 100), d=rng.randint(3, 25),
                    e=rng.randint(3, 22), er=rng.choice([1e-3, 1e-6]))
    if kind == "circuit":
        form = rng.choice(["plain", "plain", "chosen"])
        if form == "plain" and rng.random() < 0.4:
            return dict(kind=kind, n=rng.randint(8, 14),
                        depth=rng.randint(6, 10), chi=rng.choice([16, 32, 50]),
                        cutoff=1e-10, form=form, batched=False,
                        gates=rng.choice(["haar", "weak"]))
        return dict(kind=kind, n=rng.randint(16, 40),
                    depth=rng.randint(10, 20), chi=_log(rng, 48, 256),
                    cutoff=1e-8, form=form, batched=True,
                    gates=rng.choice(["haar", "haar", "weak"]))
    if kind == "batch":
        return dict(kind=kind, count=_log(rng, 4, 24),
                    chi=rng.choice([32, 64, 128]), cutoff=1e-8, form="plain")
    if kind == "expect":
        return dict(kind=kind, n=rng.randint(14, 24),
                    chi=rng.randint(96, 512), form="plain")
    if kind == "zipup":
        return dict(kind=kind, n=rng.randint(10, 24), chi=_log(rng, 24, 128),
                    cutoff=1e-10)
    return dict(kind=kind, nb=_log(rng, 300, 4096),
                minibatch=rng.choice([128, 256, 512]),
                steps=_log(rng, 8, 128))


# ---------------------------------------------------------------------------
# inputs

def _crand(seed, *shape):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal(shape) +
            1j * rng.standard_normal(shape)) / np.sqrt(2.0)


def _pair_arrays(case, seed):
    a, b, c, d = case["a"], case["b"], case["c"], case["d"]
    return _crand([seed, 1], a, b, c), _crand([seed, 2], c, b, d)


def _svd_arrays(case, seed):
    """Two tensors whose shared leg carries a decaying spectrum, as the legs
    of a truncated network do."""
    a, b, c, d, e = (case[k] for k in "abcde")
    fall = np.exp(-12.0 * np.arange(c) / c)
    A = _crand([seed, 1], a, b, c) * fall
    B = fall[:, None, None] * _crand([seed, 2], c, d, e)
    return A / np.linalg.norm(A), B / np.linalg.norm(B)


def _network(case, seed):
    net, _ = W.qft_expectation_network(case["n"], seed)
    if case["order"] == "treewidth":
        NG.optimize_contraction_order(net)
    return net


def _layers(case, seed):
    if case["gates"] == "weak":
        return C.weak_brickwall_layers(case["n"], case["depth"], seed)
    return C.brickwall_layers(case["n"], case["depth"], seed)


def _batch_sizes(case):
    """(n, depth, chi) of every circuit of the batch, the case's own: 16 to
    48 qubits, depth 8 to 24, caps up to the case's."""
    rng = np.random.default_rng(case["count"])
    return [(int(rng.integers(16, 49)), int(rng.integers(8, 25)),
             int(rng.choice([x for x in (32, 64, 128) if x <= case["chi"]])))
            for _ in range(case["count"])]


def _batch_circuits(case, seed):
    return [(n, depth, chi, C.brickwall_layers(n, depth, seed * 1009 + i))
            for i, (n, depth, chi) in enumerate(_batch_sizes(case))]


def _bits(n, seed):
    if n <= 12:
        k = np.arange(2 ** n)
        return ((k[:, None] >> np.arange(n)) & 1).astype(np.uint8)
    return C.random_bitstrings(n, 256, seed)


def _tfim(case, seed):
    n = case["n"]
    return (H.random_mps_tensors(n, case["chi"], seed),
            H.tfim_mpo(n, 1.0, H.tfim_fields(n, seed)))


def _training_set(case, seed):
    """Features as the library gathers them (a normalised, falling spectrum,
    operator-Schmidt coefficients, the bond's place and sizes) and kept
    ranks."""
    nb = case["nb"]
    rng = np.random.default_rng(seed)
    X = np.zeros((72, nb), dtype=np.float32)
    s = np.exp(-np.arange(64)[:, None] * rng.uniform(0.01, 0.4, nb)[None, :])
    X[:64] = s / np.linalg.norm(s, axis=0)
    X[64:68] = -np.sort(-rng.uniform(0, 1.5, (4, nb)), axis=0)
    X[68:72] = rng.uniform(0, 1, (4, nb))
    T = (0.5 * X[69] + 0.5 * X[71]) * (1.0 - np.exp(-3 * X[1] / X[0]))
    return X, T.astype(np.float32)


def _device(a):
    """A complex128 array on the GPU, column-major."""
    return torch.from_numpy(np.ascontiguousarray(
        np.asarray(a).reshape(-1, order="F"))).cuda()


def _ptr(t):
    return ctypes.cast(t.data_ptr(), ctypes.POINTER(ctypes.c_double))


def prepare(case, seed):
    kind = case["kind"]
    ctx = default_context()
    st = {"case": case, "ctx": ctx}
    if kind == "pair":
        A, B = _pair_arrays(case, seed)
        st["A"], st["B"] = np.asfortranarray(A), np.asfortranarray(B)
    elif kind == "theta":
        l, m, r = case["l"], case["m"], case["r"]
        st["A"] = _device(_crand([seed, 1], l, 2, m))
        st["B"] = _device(_crand([seed, 2], m, 2, r))
        st["out"] = torch.empty(4 * l * r, dtype=torch.complex128,
                                device="cuda")
        st["dA"] = np.array([l, 2, m], dtype=np.int64)
        st["dB"] = np.array([m, 2, r], dtype=np.int64)
        st["la"] = np.array([3], dtype=np.int32)
        st["lb"] = np.array([1], dtype=np.int32)
        st["perm"] = np.array([int(x) for x in case["order"]],
                              dtype=np.int32)
        torch.cuda.synchronize()
    elif kind == "net":
        st["net"] = _network(case, seed)
    elif kind == "svd":
        A, B = _svd_arrays(case, seed)
        st["A"], st["B"] = np.asfortranarray(A), np.asfortranarray(B)
    elif kind == "circuit":
        st["layers"] = _layers(case, seed)
        st["bits"] = _bits(case["n"], seed)
    elif kind == "batch":
        st["circuits"] = _batch_circuits(case, seed)
        st["bits"] = [_bits(c[0], seed)[:64] for c in st["circuits"]]
    elif kind == "expect":
        sites, mpo = _tfim(case, seed)
        st["psi"] = DeviceMPS(case["n"], case["chi"], ctx)
        st["psi"].set_sites(sites)
        st["mpo"] = DeviceMPO(mpo, ctx)
    elif kind == "zipup":
        sites, mpo = _tfim(case, seed)
        st["psi"] = DeviceMPS(case["n"], case["chi"], ctx)
        st["psi"].set_sites(sites)
        st["mpo"] = DeviceMPO(mpo, ctx)
        st["out"] = DeviceMPS(case["n"], case["chi"], ctx)
        st["bits"] = _bits(case["n"], seed)
    elif kind == "mlp":
        st["X"], st["T"] = _training_set(case, seed)
        st["init"] = learned.init_params(seed)
    ctx.sync()
    return st


# ---------------------------------------------------------------------------
# one pass

def _table(spectra, chi):
    """The bond spectra as rows of a table, zeros behind each."""
    out = np.zeros((len(spectra), chi))
    for row, s in zip(out, spectra):
        row[:len(s)] = s
    return out


def _state_values(dev, bits):
    return {"dims": dev.bond_dims(),
            "spectra": _table([dev.bond_spectrum(b)
                               for b in range(1, dev.n)], dev.cap),
            "amplitudes": dev.amplitudes(bits), "z": dev.expect_z()}


def run(state):
    case, ctx = state["case"], state["ctx"]
    kind = case["kind"]
    if kind == "pair":
        return ops.contract_pair(state["A"], state["B"], [3, 2], [1, 2])
    if kind == "theta":
        L.check(L.load().qtn_contract_pair_dev(
            ctx.handle, _ptr(state["A"]), 3, L.i64ptr(state["dA"]),
            _ptr(state["B"]), 3, L.i64ptr(state["dB"]), 1,
            L.i32ptr(state["la"]), L.i32ptr(state["lb"]),
            L.i32ptr(state["perm"]), _ptr(state["out"])))
        return state["out"]
    if kind == "net":
        return contract(state["net"])
    if kind == "svd":
        return ops.contract_svd(state["A"], state["B"], 3, 1, case["er"])
    if kind == "circuit":
        dev = DeviceMPS(case["n"], case["chi"], ctx)
        rec = []
        dev.run_layers(state["layers"], case["cutoff"], case["chi"],
                       FORMS[case["form"]], batched=case["batched"],
                       record=rec)
        out = _state_values(dev, state["bits"])
        out["kept"] = np.array([k for _, k, _ in rec], dtype=np.int64)
        out["weight"] = 1.0 - np.array([d for _, _, d in rec])
        dev.free()
        return out
    if kind == "batch":
        circs = state["circuits"]
        devs = [DeviceMPS(n, chi, ctx) for n, _, chi, _ in circs]
        run_circuits(devs, [c[3] for c in circs], [c[2] for c in circs],
                     case["cutoff"], FORMS[case["form"]])
        vals = [_state_values(d, b) for d, b in zip(devs, state["bits"])]
        for d in devs:
            d.free()
        # amplitudes of different circuits have different sizes: each by its
        # own power of two
        return {"dims": np.concatenate([v["dims"] for v in vals]),
                "spectra": np.concatenate([v["spectra"].ravel()
                                           for v in vals]),
                "amplitudes": np.concatenate(
                    [v["amplitudes"] * 2.0 ** (0.5 * c[0])
                     for v, c in zip(vals, circs)]),
                "z": np.concatenate([v["z"] for v in vals])}
    if kind == "expect":
        e = state["psi"].expect_mpo(state["mpo"], FORMS[case["form"]])
        return np.array([e])
    if kind == "zipup":
        nrm = state["psi"].apply_mpo(state["mpo"], case["cutoff"],
                                     case["chi"], state["out"])
        out = _state_values(state["out"], state["bits"])
        out["norm"] = nrm
        return out
    mlp = learned.RankMLP(state["init"], ctx=ctx)
    loss = mlp.train(state["X"], state["T"], steps=case["steps"],
                     minibatch=case["minibatch"], lr=2e-3)
    out = {"loss": loss, "params": mlp.params()}
    mlp.free()
    return out


# ---------------------------------------------------------------------------
# the work a pass cannot do without

def _bond_dims(n, chi):
    return [min(chi, 2 ** min(j, n - j)) for j in range(n + 1)]


def _svd_flops(m, n):
    """Thin complex SVD with vectors, Golub & Reinsch's count."""
    m, n = max(m, n), min(m, n)
    return 4 * (14 * m * n * n + 8 * n ** 3)


def _circuit_work(n, depth, chi):
    """Bonds as full-rank gates leave them: a gate multiplies what its bond
    can hold by four, up to the cap and the chain's own limit."""
    lim = _bond_dims(n, chi)
    d = [1] * (n + 1)
    by = fl = 0
    for layer in range(depth):
        for w in range(1 if layer % 2 == 0 else 2, n, 2):
            a, m, b = d[w - 1], d[w], d[w + 1]
            fl += 16 * a * m * b * 2 + 128 * a * b + _svd_flops(2 * a, 2 * b)
            k = min(lim[w], 2 * a, 2 * b)
            by += 16 * 2 * (a * m + m * b + a * k + k * b)
            d[w] = k
    return by, fl


def _net_sizes(case):
    """(bytes, flops) of the network's pairwise steps in its order."""
    net = _network(case, 1)
    labels = [list(x) for x in contract_rep(net)]
    size = {x: s for t, l in zip(net.tensors, labels)
            for x, s in zip(l, t.data.shape)}
    by = 16 * sum(t.data.size for t in net.tensors)
    fl = 0
    live = [set(x) for x in labels]
    for lab in sorted(x for x in size if x > 0):
        two = [t for t in live if lab in t]
        if len(two) < 2:
            continue
        a, b = two
        fl += 8 * math.prod(size[x] for x in a | b)
        live = [t for t in live if t is not a and t is not b] + [a ^ b]
    return by, fl


def work(case):
    kind = case["kind"]
    if kind == "pair":
        a, b, c, d = case["a"], case["b"], case["c"], case["d"]
        return {"bytes": 16 * (a * b * c + c * b * d + a * d),
                "flops": 8 * a * b * c * d}
    if kind == "theta":
        l, m, r = case["l"], case["m"], case["r"]
        return {"bytes": 16 * (2 * l * m + 2 * m * r + 4 * l * r),
                "flops": 8 * 4 * l * m * r}
    if kind == "net":
        by, fl = _net_sizes(case)
        return {"bytes": by, "flops": fl}
    if kind == "svd":
        a, b, c, d, e = (case[k] for k in "abcde")
        return {"bytes": 16 * (a * b * c + c * d * e + a * b * d * e),
                "flops": _svd_flops(a * b, c) + _svd_flops(c, d * e) +
                8 * a * b * c * d * e}
    if kind == "circuit":
        by, fl = _circuit_work(case["n"], case["depth"], case["chi"])
        return {"bytes": by, "flops": fl}
    if kind == "batch":
        by = fl = 0
        for n, depth, chi in _batch_sizes(case):
            b, f = _circuit_work(n, depth, chi)
            by, fl = by + b, fl + f
        return {"bytes": by, "flops": fl}
    if kind in ("expect", "zipup"):
        d = _bond_dims(case["n"], case["chi"])
        D = 3
        by = fl = 0
        for j in range(case["n"]):
            a, b = d[j], d[j + 1]
            by += 16 * 2 * a * b
            fl += 8 * 2 * a * a * D * b + 8 * 2 * a * b * D * b
            if kind == "zipup":
                fl += _svd_flops(2 * a, 3 * b) + _svd_flops(a, 2 * b)
                by += 16 * 2 * a * b
        return {"bytes": by, "flops": fl}
    weights = 72 * 128 + 128 * 128 + 128
    return {"bytes": 4 * (73 * min(case["nb"],
                                   case["steps"] * case["minibatch"]) +
                          6 * case["steps"] * weights),
            "flops": 6 * weights * case["steps"] * min(case["minibatch"],
                                                       case["nb"])}


# ---------------------------------------------------------------------------
# the same outputs from plain numpy and torch in 64 bits

def _rank(s, er):
    """The fewest leading values whose tail has 2-norm <= er."""
    tail = np.sqrt(np.cumsum(s[::-1] ** 2))[::-1]
    return int(np.sum(tail > er))


def _svd_keep(M, cutoff, chi):
    U, S, V = np.linalg.svd(M, full_matrices=False)
    k = _rank(S, cutoff * np.linalg.norm(S))
    return U, S, V, min(k, chi) if chi else k


class _Chain:
    """A matrix-product state in the right-canonical gauge with its bond
    spectra (Hastings, J. Math. Phys. 50, 095207); sites (left, 2, right)."""

    def __init__(self, n):
        one = np.zeros((1, 2, 1), dtype=np.complex128)
        one[0, 0, 0] = 1.0
        self.B = [one.copy() for _ in range(n)]
        self.lam = [np.ones(1) for _ in range(n + 1)]

    def one(self, w, u):
        self.B[w - 1] = np.tensordot(u, self.B[w - 1], (1, 1)).transpose(
            1, 0, 2)

    def two(self, w, g, cutoff, chi):
        A, B = self.B[w - 1], self.B[w]
        l, r = A.shape[0], B.shape[2]
        t = np.tensordot(A, B, (2, 0)).transpose(2, 1, 0, 3)  # t, s, l, r
        t = (g @ t.reshape(4, l * r)).reshape(2, 2, l, r)
        phi = t.transpose(2, 1, 3, 0).reshape(2 * l, 2 * r)  # (l s)(r t)
        _, S, V, k = _svd_keep(np.repeat(self.lam[w - 1], 2)[:, None] * phi,
                               cutoff, chi)
        nrm = np.linalg.norm(S[:k])
        self.B[w] = V[:k].reshape(k, r, 2).transpose(0, 2, 1)
        self.B[w - 1] = (phi @ V[:k].conj().T / nrm).reshape(l, 2, k)
        self.lam[w] = S[:k] / nrm
        return k, (nrm / np.linalg.norm(S)) ** 2

    def values(self, bits, chi):
        n = len(self.B)
        v = np.ones((len(bits), 1), dtype=np.complex128)
        for j, B in enumerate(self.B):
            nv = np.empty((len(bits), B.shape[2]), dtype=np.complex128)
            for s in (0, 1):
                at = bits[:, j] == s
                nv[at] = v[at] @ B[:, s, :]
            v = nv
        right = [None] * n + [np.ones((1, 1), dtype=np.complex128)]
        for j in range(n - 1, -1, -1):
            B = self.B[j]
            right[j] = sum(B[:, s] @ right[j + 1] @ B[:, s].conj().T
                           for s in (0, 1))
        left = np.ones((1, 1), dtype=np.complex128)
        z = np.empty(n)
        for j, B in enumerate(self.B):
            e = [B[:, s].conj().T @ left @ B[:, s] for s in (0, 1)]
            w = [np.sum(x.T * right[j + 1]).real for x in e]
            z[j] = (w[0] - w[1]) / (w[0] + w[1])
            left = e[0] + e[1]
        return {"dims": np.array([1] + [B.shape[2] for B in self.B]),
                "spectra": _table(self.lam[1:-1], chi),
                "amplitudes": v[:, 0], "z": z}


def _run_chain(n, layers, cutoff, chi):
    st = _Chain(n)
    kept, weight = [], []
    for singles, pairs in layers:
        for w, u in singles:
            st.one(w, u)
        for w, g in pairs:
            k, f = st.two(w, g, cutoff, chi)
            kept.append(k)
            weight.append(f)
    return st, kept, weight


def _zipup(sites, mpo, cutoff, chi):
    """Zip-up from the left of a right-canonical chain, then a truncating
    SVD sweep back (Stoudenmire & White, New J. Phys. 12, 055026)."""
    B = [b.copy() for b in sites]
    n = len(B)
    for j in range(n - 1, 0, -1):  # right-canonical by QR
        a, _, b = B[j].shape
        Q, R = np.linalg.qr(B[j].reshape(a, 2 * b).conj().T)
        B[j] = Q.conj().T.reshape(-1, 2, b)
        B[j - 1] = np.tensordot(B[j - 1], R.conj().T, (2, 0))
    B[0] = B[0] / np.linalg.norm(B[0])
    carry = np.ones((1, 1, 1), dtype=np.complex128)
    out = []
    for j in range(n):
        t = np.tensordot(carry, B[j], (2, 0))            # k, D, s, b
        t = np.tensordot(t, mpo[j], ((1, 2), (0, 2)))    # k, b, s', D'
        t = t.transpose(0, 2, 3, 1)                      # k, s', D', b
        k, _, D, b = t.shape
        if j == n - 1:
            out.append(t.reshape(k, 2, D * b))
            break
        U, S, V, kk = _svd_keep(t.reshape(2 * k, D * b), cutoff, chi)
        out.append(U[:, :kk].reshape(k, 2, kk))
        carry = (S[:kk, None] * V[:kk]).reshape(kk, D, b)
    st = _Chain(n)
    st.B = out
    for j in range(n - 1, 0, -1):
        a, _, b = st.B[j].shape
        U, S, V, k = _svd_keep(st.B[j].reshape(a, 2 * b), cutoff, chi)
        st.B[j] = V[:k].reshape(k, 2, b)
        st.lam[j] = S[:k] / np.linalg.norm(S[:k])
        st.B[j - 1] = np.tensordot(st.B[j - 1], U[:, :k] * S[:k], (2, 0))
    nrm = float(np.linalg.norm(st.B[0]))
    st.B[0] = st.B[0] / nrm
    return st, nrm


def _expect(sites, mpo):
    """<psi|W|psi> / <psi|psi> by one environment sweep, rescaled site by
    site, in complex128 on the GPU."""
    E = torch.ones((1, 1, 1), dtype=torch.complex128, device="cuda")
    N = torch.ones((1, 1), dtype=torch.complex128, device="cuda")
    for B, Wj in zip(sites, mpo):
        B = torch.from_numpy(np.ascontiguousarray(B)).cuda()
        a, _, b = B.shape
        Bc = B.conj().resolve_conj().reshape(2 * a, b).t().contiguous()
        D, De = Wj.shape[0], Wj.shape[3]
        t = [[E[:, d].contiguous() @ B[:, s].contiguous() for s in (0, 1)]
             for d in range(D)]                        # (a', b)
        nxt = []
        for e in range(De):
            u = torch.zeros((a, 2, b), dtype=torch.complex128, device="cuda")
            for o in (0, 1):
                for d in range(D):
                    for s in (0, 1):
                        if Wj[d, o, s, e]:
                            u[:, o] += complex(Wj[d, o, s, e]) * t[d][s]
            nxt.append(Bc @ u.reshape(2 * a, b))
        v = torch.stack([N @ B[:, s].contiguous() for s in (0, 1)], 1)
        N = Bc @ v.reshape(2 * a, b)
        f = float(N.abs().max())
        E = torch.stack(nxt, 1) / f
        N = N / f
    return complex(E[0, 0, 0]) / complex(N[0, 0])


def _erf(x):
    return torch.erf(torch.from_numpy(x)).numpy()


def _train(case, seed):
    X, T = _training_set(case, seed)
    X, T = X.astype(np.float64), T.astype(np.float64)
    X[:64] = np.log10(np.maximum(X[:64], 1e-16)) / 8.0
    p = learned.init_params(seed).astype(np.float64)
    nin, wd = 72, 128
    cut = np.cumsum([0, wd * nin, wd, wd * wd, wd, wd, 1])
    shape = [(wd, nin), (wd, 1), (wd, wd), (wd, 1), (1, wd), (1, 1)]
    nb, mb = case["nb"], min(case["minibatch"], case["nb"])
    m1, m2 = np.zeros_like(p), np.zeros_like(p)
    loss = []

    def gelu(z):
        return 0.5 * z * (1.0 + _erf(z / np.sqrt(2.0)))

    def slope(z):
        return 0.5 * (1.0 + _erf(z / np.sqrt(2.0))) + \
            z * np.exp(-0.5 * z * z) / np.sqrt(2.0 * np.pi)

    for t in range(case["steps"]):
        at = (t * mb) % nb
        x, y = X[:, at:at + mb], T[at:at + mb]
        W1, b1, W2, b2, W3, b3 = (
            p[cut[i]:cut[i + 1]].reshape(shape[i], order="F")
            for i in range(6))
        z1 = W1 @ x + b1
        a1 = gelu(z1)
        z2 = W2 @ a1 + b2
        a2 = gelu(z2)
        r = (W3 @ a2 + b3)[0] - y
        loss.append(np.mean(r * r))
        d3 = (2.0 * r / r.size)[None, :]
        d2 = (W3.T @ d3) * slope(z2)
        d1 = (W2.T @ d2) * slope(z1)
        g = np.concatenate([v.reshape(-1, order="F") for v in (
            d1 @ x.T, d1.sum(1), d2 @ a1.T, d2.sum(1), d3 @ a2.T,
            d3.sum(1))])
        m1 = 0.9 * m1 + 0.1 * g
        m2 = 0.999 * m2 + 0.001 * g * g
        p = p - 2e-3 * (m1 / (1 - 0.9 ** (t + 1))) / (
            np.sqrt(m2 / (1 - 0.999 ** (t + 1))) + 1e-8)
    return {"loss": np.array(loss), "params": p}


def exact(case, seed):
    kind = case["kind"]
    if kind == "pair":
        A, B = _pair_arrays(case, seed)
        return np.tensordot(A, B, ((2, 1), (0, 1)))
    if kind == "theta":
        l, m, r = case["l"], case["m"], case["r"]
        t = np.tensordot(_crand([seed, 1], l, 2, m),
                         _crand([seed, 2], m, 2, r), (2, 0))
        t = t.transpose([int(x) - 1 for x in case["order"]])
        return t.reshape(-1, order="F")
    if kind == "net":
        net = _network(case, seed)
        live = [(t.data, list(x)) for t, x in
                zip(net.tensors, contract_rep(net))]
        for lab in sorted({x for _, l in live for x in l if x > 0}):
            two = [i for i, (_, l) in enumerate(live) if lab in l]
            if not two:
                continue
            (a, la), (b, lb) = live[two[0]], live[two[1]]
            both = [x for x in la if x in lb]
            c = np.tensordot(a, b, ([la.index(x) for x in both],
                                    [lb.index(x) for x in both]))
            lc = [x for x in la if x not in both] + \
                [x for x in lb if x not in both]
            live = [v for i, v in enumerate(live) if i not in two]
            live.append((c, lc))
        out = np.array(1.0 + 0j)
        for c, _ in live:
            out = out * c
        return out
    if kind == "svd":
        A, B = _svd_arrays(case, seed)
        a, b, c = A.shape
        U1, S1, V1 = np.linalg.svd(A.reshape(a * b, c), full_matrices=False)
        k1 = _rank(S1, case["er"])
        U2, S2, V2 = np.linalg.svd(B.reshape(c, -1), full_matrices=False)
        k2 = _rank(S2, case["er"])
        mid = (S1[:k1, None] * V1[:k1]) @ (U2[:, :k2] * S2[:k2])
        return ((U1[:, :k1] @ mid) @ V2[:k2]).reshape(
            a, b, B.shape[1], B.shape[2])
    if kind == "circuit":
        st, kept, weight = _run_chain(case["n"], _layers(case, seed),
                                      case["cutoff"], case["chi"])
        out = st.values(_bits(case["n"], seed), case["chi"])
        out["kept"] = np.array(kept, dtype=np.int64)
        out["weight"] = np.array(weight)
        return out
    if kind == "batch":
        vals = []
        for n, _, chi, layers in _batch_circuits(case, seed):
            st, _, _ = _run_chain(n, layers, case["cutoff"], chi)
            v = st.values(_bits(n, seed)[:64], chi)
            v["spectra"] = v["spectra"].ravel()
            v["amplitudes"] = v["amplitudes"] * 2.0 ** (0.5 * n)
            vals.append(v)
        return {k: np.concatenate([v[k] for v in vals]) for k in vals[0]}
    if kind == "expect":
        return np.array([_expect(*_tfim(case, seed))])
    if kind == "zipup":
        st, nrm = _zipup(*_tfim(case, seed), case["cutoff"], case["chi"])
        out = st.values(_bits(case["n"], seed), case["chi"])
        out["norm"] = nrm
        return out
    return _train(case, seed)
