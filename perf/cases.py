"""The workloads that this library's speed is measured on.

Each case is one call (or one training step) that a program using the library
makes on the GPU, at the sizes of its configurations and examples: permanents
of matrix batches, SLOS strong simulation of one input and of an input tree,
exact sampling, phase gradients, Gurvits estimates, and the learned sampler's
training step and chain.  Inputs come from the seed alone; `exact` restates
each result in float64 with plain torch.

  listed()             the named cases
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  what a program holds before the call
  run(state)           one pass through the public entry points
  work(case)           bytes and operations a pass cannot do without
  exact(case, seed)    run's result in float64 without the library, or None
"""
from __future__ import annotations

import itertools
import math

import numpy as np
import torch

DEV = "cuda"
MESH_KEYS = ("m", "n", "targets", "sets", "weighted")


def listed():
    return [
        # all 12,376 outputs of 6 photons in 12 modes through their permanents
        # (what the Naive backend batches): the smallest orders, launch-bound
        {"name": "perm_n6_b12376", "kind": "perm", "nlo": 6, "nhi": 6, "count": 12376, "m": 12},
        # the headline batch: 4,096 order-20 submatrices of a 64-mode unitary
        {"name": "perm_n20_b4096", "kind": "perm", "nlo": 20, "nhi": 20, "count": 4096, "m": 64},
        # outputs of different photon numbers in one launch: orders 12..24 mixed
        {"name": "perm_mixed_n12_24_b1000", "kind": "perm", "nlo": 12, "nhi": 24, "count": 1000, "m": 64},
        # an everyday strong simulation, one circuit of a parameter scan: short
        # layers, where a pass is launches and latency
        {"name": "slos_m12_n6", "kind": "slos", "m": 12, "n": 6, "coefs": False, "herald": 0},
        # the largest strong simulation of the configurations: 92,561,040 outputs
        {"name": "slos_m24_n10", "kind": "slos", "m": 24, "n": 10, "coefs": False, "herald": 0},
        # a noisy source: 8 photons in 20 modes with every one- and two-photon
        # loss, 37 inputs sharing one tree of layers
        {"name": "slos_tree_m20_n8_loss2", "kind": "tree", "m": 20, "n": 8, "lost": 2},
        # exact sampling at the largest configured circuit
        {"name": "sample_m60_n20_20000", "kind": "sample", "m": 60, "n": 20, "count": 20000, "lost": 0},
        # a noisy source's sample pools: 37 inputs x 2,000 samples in one call
        {"name": "sample_m20_n8_37x2000", "kind": "sample", "m": 20, "n": 8, "count": 2000, "lost": 2},
        # a variational step over every output (462 weighted outputs of 6
        # photons in 6 modes): loss, and its gradient for 256 parameter sets
        {"name": "mesh_m6_n6_t462_b256", "kind": "mesh", "m": 6, "n": 6, "targets": 462, "sets": 256,
         "weighted": True},
        # approximate amplitudes of 30 photons in 60 modes, a million draws each
        {"name": "gurvits_n30_b64", "kind": "gurvits", "n": 30, "m": 60, "count": 64, "iters": 1000000},
        # one optimiser step of the learned proposal on 2,048 sequences
        {"name": "train_m60_n20_b2048", "kind": "train", "m": 60, "n": 20, "batch": 2048},
        # the learned sampler's chain: propose, score by permanents, accept
        {"name": "chain_m60_n20_100000", "kind": "chain", "m": 60, "n": 20, "count": 100000},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["perm", "perm", "perm", "slos", "slos", "tree", "sample", "sample", "mesh", "mesh", "gurvits",
                       "train", "chain"])
    while True:
        if kind == "perm":     # single and mixed orders, one matrix to many
            nlo = rng.randint(2, 24)
            nhi = rng.choice([nlo, rng.randint(nlo, 24)])
            case = {"kind": "perm", "nlo": nlo, "nhi": nhi, "count": _log_int(rng, 1, 20000),
                    "m": max(nhi, rng.choice([24, 64]))}
            ok = work(case)["flops"] <= 3.4e11
        elif kind == "slos":   # probabilities or coefficients, with or without heralded modes
            case = {"kind": "slos", "m": rng.randint(4, 26), "n": rng.randint(2, 10), "coefs": rng.random() < 0.4,
                    "herald": rng.choice([0, 0, 1, 2])}
            # heralds compute the outputs that match; two modes at least stay free, and a photon
            ok = (_fock(case["m"], case["n"]) <= (45_000_000 if case["coefs"] else 93_000_000)
                  and (case["herald"] == 0 or (case["m"] - case["herald"] >= 3 and not case["coefs"]
                                               and case["n"] > 2)))
        elif kind == "tree":
            n = rng.randint(3, 8)
            case = {"kind": "tree", "m": rng.randint(n, 20), "n": n, "lost": rng.choice([1, 2])}
            ok = True
        elif kind == "sample":
            n = rng.randint(2, 20)
            case = {"kind": "sample", "m": rng.randint(n, 60), "n": n, "count": _log_int(rng, 1, 50000),
                    "lost": rng.choice([0, 0, 1, 2]) if n <= 10 else 0}
            ok = work(case)["flops"] <= work(listed()[6])["flops"] * 1.001
        elif kind == "mesh":
            m, n = rng.randint(4, 16), rng.randint(1, 6)
            case = {"kind": "mesh", "m": m, "n": n, "targets": min(_log_int(rng, 1, 512), _fock(m, n)),
                    "sets": _log_int(rng, 1, 1024), "weighted": rng.random() < 0.5}
            ok = work(case)["flops"] <= 8 * work(listed()[8])["flops"]
        elif kind == "gurvits":
            n = rng.randint(2, 40)
            case = {"kind": "gurvits", "n": n, "m": max(n, 60), "count": rng.randint(1, 64),
                    "iters": _log_int(rng, 10000, 1000000)}
            ok = work(case)["flops"] <= work(listed()[9])["flops"]
        elif kind == "train":
            n = rng.randint(4, 20)
            case = {"kind": "train", "m": rng.randint(n, 60), "n": n, "batch": _log_int(rng, 128, 2048)}
            ok = True
        else:
            n = rng.randint(4, 20)
            case = {"kind": "chain", "m": rng.randint(n, 60), "n": n, "count": _log_int(rng, 1000, 100000)}
            ok = True
        if ok:
            return case


# ------------------------------------------------------------------ inputs

def _fock(m, n):
    return math.comb(m + n - 1, n)


def _haar(m, rng):
    q, r = np.linalg.qr(rng.randn(m, m) + 1j * rng.randn(m, m))
    return q @ np.diag(np.sign(np.diagonal(r).real))


def _orders(case):
    # the batch's orders are the case's own, whatever the seed: a plan is for them
    lo, hi, count = case["nlo"], case["nhi"], case["count"]
    return np.random.RandomState(lo * 1000 + hi).randint(lo, hi + 1, size=count).astype(np.int32)


def _matrices(case, seed):
    """The batch's submatrices of one Haar unitary, packed back to back."""
    rng = np.random.RandomState(seed)
    m, orders = case["m"], _orders(case)
    U = _haar(m, rng)
    flat = np.empty(int((orders.astype(np.int64) ** 2).sum()), dtype=np.complex128)
    at = 0
    rows = rng.rand(len(orders), m).argsort(axis=1)
    cols = rng.rand(len(orders), m).argsort(axis=1)
    for n in np.unique(orders):
        idx = np.nonzero(orders == n)[0]
        sub = U[rows[idx, :n][:, :, None], cols[idx, :n][:, None, :]].reshape(len(idx), -1)
        if len(idx) == len(orders):
            flat[:] = sub.reshape(-1)
        else:
            start = np.concatenate([[0], np.cumsum(orders.astype(np.int64) ** 2)[:-1]])[idx]
            flat[start[:, None] + np.arange(n * n)] = sub
    return orders, flat


def _single_photons(m, n):
    return [1] * n + [0] * (m - n)


def _loss_inputs(m, n, lost):
    base = _single_photons(m, n)
    rows = [base]
    for k in range(1, lost + 1):
        for drop in itertools.combinations(range(n), k):
            rows.append([0 if i in drop else v for i, v in enumerate(base)])
    return rows


def _herald(case):
    """One photon on each of the last modes, the reference's herald shape."""
    cond = [-1] * case["m"]
    for q in range(case["herald"]):
        cond[case["m"] - 1 - q] = q % 2
    return cond


def _mesh_inputs(case, seed):
    rng = np.random.RandomState(seed)
    m, n = case["m"], case["n"]
    phases = rng.uniform(0, 2 * math.pi, size=(case["sets"], m * (m - 1)))
    # a random output list without repetition, in rank order
    seqs = set()
    if case["targets"] * 2 >= _fock(m, n):
        every = list(itertools.combinations_with_replacement(range(m), n))
        seqs = sorted(every[i] for i in rng.permutation(len(every))[:case["targets"]])
    else:
        while len(seqs) < case["targets"]:
            seqs.add(tuple(sorted(rng.randint(0, m, size=n).tolist())))
        seqs = sorted(seqs)
    targets = np.zeros((len(seqs), m), dtype=np.int32)
    for k, s in enumerate(seqs):
        for q in s:
            targets[k, q] += 1
    w = None
    if case["weighted"]:
        w = rng.rand(len(seqs)) + 1e-3 * np.arange(len(seqs))
        w = 200 * (w - w.mean()) / w.std() if len(seqs) > 1 else np.ones(1)
    # the input photons, in the first modes (two in a mode when n > m)
    occ = [n // m + (1 if i < n % m else 0) for i in range(m)]
    return phases, occ, targets, w


def _gurvits_matrices(case, seed):
    rng = np.random.RandomState(seed)
    U = _haar(case["m"], rng)
    n = case["n"]
    return [np.ascontiguousarray(U[np.sort(rng.choice(case["m"], n, replace=False))][:, :n])
            for _ in range(case["count"])]


def _sequences(rng, count, m, n):
    """Uniform bosonic outputs (the Haar average of boson sampling) as sorted mode sequences."""
    sel = rng.rand(count, m + n - 1).argsort(axis=1)[:, :n]
    return (np.sort(sel, axis=1) - np.arange(n)).astype(np.int32)


def _net_weights(m, n, rng, hidden=256):
    """A proposal network near the law a trained one starts from: unit p of
    the first layer passes step p on, its output row holds the log counts of
    sorted completions (uniform over Fock states); the other units carry small
    random weights."""
    W1 = 0.05 * rng.randn(hidden, m + n)
    W2 = 0.02 * rng.randn(m, hidden)
    b1 = 0.02 * rng.randn(hidden)
    b2 = 0.02 * rng.randn(m)
    W1[:n], b1[:n] = 0.0, 0.0
    for p in range(n):
        W1[p, m + p] = 1.0
        left = n - 1 - p
        W2[:, p] += [math.lgamma(m - j + left) - math.lgamma(m - j) - math.lgamma(left + 1) for j in range(m)]
        W2[:, p] -= W2[:, p].max()
    return [v.astype(np.float32) for v in (W1, b1, W2, b2)]


def _load_net(net, weights):
    for p, w in zip(net.params, weights):
        p.copy_(torch.from_numpy(w).reshape(p.shape))
    net.refresh_bf16()


# ------------------------------------------------------------------ prepare / run

def prepare(case, seed):
    kind = case["kind"]
    s = dict(case)
    if kind == "perm":
        from perceval_amd.permanent import PermanentPlan
        orders, flat = _matrices(case, seed)
        s["packed"] = torch.from_numpy(flat).to(DEV)
        s["plan"] = PermanentPlan(orders)
    elif kind == "slos":
        from perceval_amd.slos import SlosPlan
        s["U"] = torch.from_numpy(_haar(case["m"], np.random.RandomState(seed))).to(DEV)
        occ = _photons(case)
        s["plan"] = SlosPlan(occ, mask_cond=_herald(case)) if case["herald"] else SlosPlan(occ)
    elif kind == "tree":
        from perceval_amd.slos import SlosTree
        s["U"] = torch.from_numpy(_haar(case["m"], np.random.RandomState(seed))).to(DEV)
        s["tree"] = SlosTree(_loss_inputs(case["m"], case["n"], case["lost"]))
    elif kind == "sample":
        s["U"] = torch.from_numpy(_haar(case["m"], np.random.RandomState(seed))).to(DEV)
        s["inputs"] = _loss_inputs(case["m"], case["n"], case["lost"])
        s["seed"] = seed
    elif kind == "mesh":
        from perceval_amd.components import clements_mesh
        from perceval_amd.gradient import MeshProgram
        phases, s["occ"], s["outputs"], s["w"] = _mesh_inputs(case, seed)
        s["phases"] = torch.from_numpy(phases).to(DEV).requires_grad_(True)
        s["program"] = MeshProgram(clements_mesh(case["m"]))
    elif kind == "gurvits":
        s["mats"] = _gurvits_matrices(case, seed)
        s["seed"] = seed
    elif kind == "train":
        from perceval_amd.mis import ProposalNet
        rng = np.random.RandomState(seed)
        s["seqs"] = torch.from_numpy(_sequences(rng, case["batch"], case["m"], case["n"])).to(DEV)
        s["net"] = ProposalNet(case["m"], case["n"], hidden=256)
        s["weights"] = _net_weights(case["m"], case["n"], rng)
        _load_net(s["net"], s["weights"])
    elif kind == "chain":
        from perceval_amd.mis import LearnedMIS, ProposalNet
        rng = np.random.RandomState(seed)
        U = _haar(case["m"], rng)
        net = ProposalNet(case["m"], case["n"], hidden=256)
        _load_net(net, _net_weights(case["m"], case["n"], rng))
        s["mis"] = LearnedMIS(U, _single_photons(case["m"], case["n"]), net)
        s["x0"] = torch.from_numpy(_sequences(rng, 1, case["m"], case["n"])[0]).to(DEV)
        s["seed"] = seed
    return s


def _photons(case):
    # one photon per mode in the first modes; more photons than modes go round again
    m, n = case["m"], case["n"]
    return [n // m + (1 if i < n % m else 0) for i in range(m)]


def run(s):
    kind = s["kind"]
    if kind == "perm":
        return s["plan"](s["packed"])
    if kind == "slos":
        from perceval_amd.slos import COEFS, PROBS
        return s["plan"].run(s["U"], COEFS if s["coefs"] else PROBS)
    if kind == "tree":
        from perceval_amd.slos import PROBS
        return s["tree"].run(s["U"], PROBS)
    if kind == "sample":
        from perceval_amd.sampling import cc_samples_device, cc_samples_multi_device
        if len(s["inputs"]) == 1:
            return cc_samples_device(s["U"], s["inputs"][0], s["count"], seed=s["seed"])
        return cc_samples_multi_device(s["U"], s["inputs"], [s["count"]] * len(s["inputs"]), seed=s["seed"])
    if kind == "mesh":
        from perceval_amd.gradient import target_probability
        loss = target_probability(s["phases"], s["program"], s["occ"], s["outputs"], s["w"])
        (grad,) = torch.autograd.grad(loss.sum(), s["phases"])
        return {"loss": loss, "grad": grad}
    if kind == "gurvits":
        from perceval_amd.permanent import gurvits
        est, err = gurvits(s["mats"], s["iters"], seed=s["seed"])
        return {"est": est, "err": err}
    if kind == "train":
        net, seqs = s["net"], s["seqs"]
        x, lo, target = net.teacher_forcing(seqs)
        loss, grads = net.loss_and_grads(x, lo, target, 1.0 / seqs.shape[0])
        net.adam_step(grads, lr=2e-3)
        return {"loss": loss, "grads": grads, "params": net.params}
    out = s["mis"].run(s["count"], seed=s["seed"], x0_seq=s["x0"])
    return {"seq": out["seq"], "acceptance": out["acceptance"], "logw": out["logw"], "proposals": out["proposals"]}


# ------------------------------------------------------------------ work

def _glynn(n):
    """Operations of Glynn's formula in Gray-code order: n complex additions,
    n - 1 complex products and one complex addition per term."""
    return float(2 ** (n - 1)) * (8 * n - 4)


def _slos_work(m, ns, matched=None):
    """Layers written once and read once, probabilities written once."""
    nmax = max(ns)
    layers = sum(_fock(m, k) for k in range(1, nmax))
    outs = sum(_fock(m, k) for k in ns) if matched is None else matched
    if matched is not None:
        layers = min(layers, matched * nmax)
    return {"bytes": 32.0 * layers + 8.0 * outs, "flops": 8.0 * (layers + outs) * nmax}


def _multiset_terms(m, k):
    """Terms of the permanent of k output photons, repeated rows summed by
    multiplicity: the mean of prod (s_j + 1) / 2 over all k-photon outputs."""
    return _fock(2 * m, k) / _fock(m, k) / 2 if k else 1.0


def work(case):
    kind = case["kind"]
    if kind == "perm":
        orders = _orders(case).tolist()
        return {"bytes": 16.0 * sum(n * n + 1 for n in orders), "flops": sum(_glynn(n) for n in orders)}
    if kind == "slos":
        m, n, h = case["m"], case["n"], case["herald"]
        matched = None
        if h:
            matched = _fock(m - h, n - sum(c for c in _herald(case) if c > 0))
        w = _slos_work(m, [n], matched)
        if case["coefs"]:
            w["bytes"] += 8.0 * _fock(m, n)
        return w
    if kind == "tree":
        return _slos_work(case["m"], [sum(r) for r in _loss_inputs(case["m"], case["n"], case["lost"])])
    if kind == "sample":
        m = case["m"]
        flops = total = 0.0
        for r in _loss_inputs(m, case["n"], case["lost"]):
            n = sum(r)
            # photon k: its k sub-permanents share one sum of k column sums, prefix and suffix products
            flops += case["count"] * sum(_multiset_terms(m, k - 1) * 24 * k + 8 * m * k for k in range(1, n + 1))
            total += case["count"]
        return {"bytes": total * 4 * m + 16.0 * m * m, "flops": flops}
    if kind == "mesh":
        m, n, T, B = case["m"], case["n"], case["targets"], case["sets"]
        per = T * 2 ** max(0, n - 1) * 24 * n + 3 * 28.0 * m * m * (m - 1)
        return {"bytes": B * (16.0 * m * (m - 1) + 8), "flops": float(B * per)}
    if kind == "gurvits":
        n = case["n"]
        return {"bytes": 16.0 * case["count"] * n * n, "flops": float(case["count"]) * case["iters"] *
                (4 * n * n + 6 * (n - 1))}
    if kind == "train":
        m, n, R = case["m"], case["n"], case["batch"] * case["n"]
        params = 256 * (m + n + 1) + m * 257
        return {"bytes": 4.0 * R + 28.0 * params, "flops": 2.0 * R * 256 * (2 * (m + n) + 3 * m)}
    m, n, N = case["m"], case["n"], case["count"]
    return {"bytes": N * (8.0 * n + 8), "flops": N * (_multiset_terms(m, n) * (8 * n - 4) + 2.0 * n * 256 * (m + 2))}


# ------------------------------------------------------------------ exact

def _perms(A):
    """Permanents of a (b, n, n) complex128 batch by Glynn's formula, terms
    summed pairwise: low sign patterns in a table, high ones added to it."""
    b, n, _ = A.shape
    if n == 0:
        return torch.ones(b, dtype=A.dtype, device=A.device)
    if n == 1:
        return A[:, 0, 0].clone()
    low = min(n - 1, 9)

    def signs(k):
        t = torch.arange(2 ** k, device=A.device)
        s = [1.0 - 2.0 * ((t >> i) & 1).double() for i in range(k)]
        return torch.stack(s) if k else torch.zeros((0, 1), dtype=torch.float64, device=A.device)

    def table(rows, S):      # (b, n, patterns): signed sums of the rows, per column
        out = torch.zeros((b, n, S.shape[1]), dtype=A.dtype, device=A.device)
        for i in range(rows.shape[1]):
            out += rows[:, i, :, None] * S[i][None, None, :]
        return out

    Sl, Sh = signs(low), signs(n - 1 - low)
    T = table(A[:, 1:1 + low], Sl) + A[:, 0, :, None]
    H = table(A[:, 1 + low:], Sh)
    pl = Sl.prod(dim=0)
    ph = Sh.prod(dim=0) if Sh.shape[0] else torch.ones(1, dtype=torch.float64, device=A.device)
    parts = torch.empty((b, H.shape[2]), dtype=A.dtype, device=A.device)
    for h in range(H.shape[2]):
        p = T[:, 0] + H[:, 0, h, None]
        for j in range(1, n):
            p *= T[:, j] + H[:, j, h, None]
        parts[:, h] = (p * pl).sum(dim=1)
    return (parts * ph).sum(dim=1) / 2.0 ** (n - 1)


def _perms_chunked(A):
    b, n = A.shape[0], A.shape[1]
    step = max(1, int(2 ** 27 // (max(1, n) * 2 ** min(max(n - 1, 0), 9))))
    return torch.cat([_perms(A[i:i + step]) for i in range(0, b, step)]) if b else A.new_zeros(0)


def _sorted_sequences(m, n):
    """Every non-decreasing sequence of n modes, lexicographic (the order of
    descending occupation vectors), as a (count, n) tensor."""
    seq = torch.arange(m, device=DEV)[:, None]
    for _ in range(n - 1):
        reps = m - seq[:, -1]
        start = torch.cumsum(reps, 0) - reps
        seq = torch.repeat_interleave(seq, reps, dim=0)
        last = seq[:, -1] + torch.arange(seq.shape[0], device=DEV) - torch.repeat_interleave(start, reps)
        seq = torch.cat([seq, last[:, None]], dim=1)
    return seq


def _run_factorials(seq):
    """prod s_j! of every sorted sequence."""
    f = torch.ones(seq.shape[0], dtype=torch.float64, device=seq.device)
    run_len = torch.ones_like(f)
    for r in range(1, seq.shape[1]):
        run_len = torch.where(seq[:, r] == seq[:, r - 1], run_len + 1, torch.ones_like(f))
        f = f * run_len
    return f


def _slos_exact(U, occ, coefs, cond=None):
    m, n = len(occ), sum(occ)
    cols = torch.tensor([i for i, v in enumerate(occ) for _ in range(v)], device=DEV)
    pin = float(np.prod([math.factorial(v) for v in occ]))
    seq = _sorted_sequences(m, n)
    if cond is not None:
        keep = torch.ones(seq.shape[0], dtype=torch.bool, device=DEV)
        for q, c in enumerate(cond):
            if c >= 0:
                keep &= (seq == q).sum(dim=1) == c
        seq = seq[keep]
    step = max(1, int(2 ** 27 // (n * 2 ** (n - 1))))
    res = []
    for i in range(0, seq.shape[0], step):
        s = seq[i:i + step]
        p = _perms(U[s[:, :, None], cols[None, None, :]])
        f = _run_factorials(s)
        res.append(p / f if coefs else (p.real ** 2 + p.imag ** 2) / (f * pin))
    return torch.cat(res) if res else torch.zeros(0, dtype=torch.float64, device=DEV)


def _terms(case):
    """Glynn terms x columns that `exact` would form."""
    if case["kind"] == "perm":
        return sum(2.0 ** (n - 1) * n for n in _orders(case).tolist())
    ns = [case["n"]] if case["kind"] == "slos" else [sum(r) for r in
                                                     _loss_inputs(case["m"], case["n"], case["lost"])]
    return sum(_fock(case["m"], n) * 2.0 ** (n - 1) * n for n in ns)


def _mesh_exact(case, seed):
    phases, occ, targets, w = _mesh_inputs(case, seed)
    m = case["m"]
    w = torch.ones(len(targets), dtype=torch.float64) if w is None else torch.from_numpy(w)
    cols = [i for i, v in enumerate(occ) for _ in range(v)]
    pin = float(np.prod([math.factorial(v) for v in occ]))
    rows = torch.tensor([[q for q in range(m) for _ in range(t[q])] for t in targets.tolist()], device=DEV)
    norm = torch.tensor([pin * float(np.prod([math.factorial(v) for v in t])) for t in targets.tolist()],
                        dtype=torch.float64, device=DEV)
    w = w.to(DEV)
    losses, grads = [], []
    for i in range(0, case["sets"], 32):
        ph = torch.from_numpy(phases[i:i + 32]).to(DEV).requires_grad_(True)
        B = ph.shape[0]
        rowsU = [torch.eye(m, dtype=torch.complex128, device=DEV)[q].expand(B, m) for q in range(m)]
        c, sn = math.cos(math.pi / 4), math.sin(math.pi / 4)
        e = torch.polar(torch.ones_like(ph), ph)
        k = 0
        for depth in range(m):               # rectangular mesh: phase, splitter, phase, splitter
            for j in range(depth % 2, m - 1, 2):
                for _ in range(2):
                    top, low = rowsU[j] * e[:, k:k + 1], rowsU[j + 1]
                    rowsU[j], rowsU[j + 1] = c * top + 1j * sn * low, 1j * sn * top + c * low
                    k += 1
        U = torch.stack(rowsU, dim=1)
        sub = U[:, rows][..., cols]          # (B, T, n, n)
        n = sub.shape[-1]
        p = torch.zeros(sub.shape[:2], dtype=torch.complex128, device=DEV)
        for t in range(2 ** (n - 1)):
            sg = [1.0] + [1.0 - 2.0 * ((t >> b) & 1) for b in range(n - 1)]
            cs = sum(s * sub[:, :, r] for r, s in enumerate(sg))
            term = cs[..., 0]
            for q in range(1, n):
                term = term * cs[..., q]
            p = p + float(np.prod(sg)) * term
        p = p / 2.0 ** (n - 1)
        loss = (((p.real ** 2 + p.imag ** 2) / norm) * w).sum(dim=1)
        (g,) = torch.autograd.grad(loss.sum(), ph)
        losses.append(loss.detach())
        grads.append(g)
    return {"loss": torch.cat(losses), "grad": torch.cat(grads)}


def _mix64(z):
    """SplitMix64's output mixing on int64 tensors (wrapping products, logical shifts)."""
    def shr(v, k):
        return (v >> k) & ((1 << (64 - k)) - 1)
    z = z + (0x9E3779B97F4A7C15 - 2 ** 64)
    z = (z ^ shr(z, 30)) * (0xBF58476D1CE4E5B9 - 2 ** 64)
    z = (z ^ shr(z, 27)) * (0x94D049BB133111EB - 2 ** 64)
    return z ^ shr(z, 31)


def _gurvits_exact(case, seed):
    """The estimator's mean and 99% bound over the counter-based signs: bit j
    of draw s of matrix b gives the sign of column j."""
    mats = np.stack(_gurvits_matrices(case, seed))
    n, N = case["n"], case["iters"]
    est, err = [], []
    for b in range(case["count"]):
        A = torch.from_numpy(mats[b]).to(DEV)
        key = _mix64(torch.tensor(seed, device=DEV) ^ _mix64(torch.tensor(b, device=DEV)))
        tot, sq = 0.0, 0.0
        for i in range(0, N, 1 << 19):
            s = torch.arange(i, min(N, i + (1 << 19)), device=DEV)
            bits = _mix64(key + s * (0x9E3779B97F4A7C15 - 2 ** 64))
            x = torch.stack([1.0 - 2.0 * ((bits >> j) & 1).double() for j in range(n)])     # (n, draws)
            y = torch.complex(A.real.contiguous() @ x, A.imag.contiguous() @ x)
            p = y[0]
            for j in range(1, n):
                p = p * y[j]
            p = p * x.prod(dim=0)
            tot = tot + p.sum()
            sq = sq + (p.real ** 2 + p.imag ** 2).sum()
        mean = tot / N
        var = (sq / N - (mean.real ** 2 + mean.imag ** 2)).clamp(min=0.0)
        est.append(mean)
        err.append(2.5758293035489004 * torch.sqrt(var / N))
    return {"est": torch.stack(est).cpu().numpy(), "err": torch.stack(err).cpu().numpy()}


def _train_exact(case, seed):
    """One step of the network in float64: products with the bf16 copies of
    the weights, as the network defines them, then Adam from zero moments."""
    rng = np.random.RandomState(seed)
    m, n = case["m"], case["n"]
    seqs = torch.from_numpy(_sequences(rng, case["batch"], m, n)).to(DEV).long()
    W1, b1, W2, b2 = (torch.from_numpy(v).to(DEV) for v in _net_weights(m, n, rng))
    W1b, W2b = W1.bfloat16().double(), W2.bfloat16().double()
    B = seqs.shape[0]
    x = torch.zeros((B, n, m + n), dtype=torch.float64, device=DEV)
    for p in range(n):
        x[:, p, m + p] = 1.0
        if p:
            x[:, p, :m] = x[:, p - 1, :m].scatter_add(1, seqs[:, p - 1:p],
                                                      torch.ones((B, 1), dtype=torch.float64, device=DEV))
    x = x.view(B * n, m + n)
    lo = torch.cat([torch.zeros((B, 1), dtype=torch.int64, device=DEV), seqs[:, :-1]], dim=1).view(-1)
    tgt = seqs.reshape(-1)
    pre = x @ W1b.T + b1.double()
    h = pre.clamp(min=0)
    z = h @ W2b.T + b2.double()
    z = z.masked_fill(torch.arange(m, device=DEV)[None, :] < lo[:, None], -math.inf)
    logq = torch.log_softmax(z, dim=1)
    loss = -logq.gather(1, tgt[:, None])[:, 0]
    dz = logq.exp()
    dz[torch.arange(B * n, device=DEV), tgt] -= 1.0
    dz /= B
    dh = (dz @ W2b) * (h > 0)
    grads = [dh.T @ x, dh.sum(0), dz.T @ h, dz.sum(0)]
    params = []
    for w, g in zip((W1, b1, W2, b2), grads):
        m1, m2 = 0.1 * g / (1 - 0.9), 0.001 * g * g / (1 - 0.999)
        params.append(w.double() - 2e-3 * m1 / (m2.sqrt() + 1e-8))
    return {"loss": loss, "grads": grads, "params": params}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("perm", "slos", "tree") and _terms(case) > 6e10:
        return None      # minutes of plain torch
    if kind == "perm":
        orders, flat = _matrices(case, seed)
        off = np.concatenate([[0], np.cumsum(orders.astype(np.int64) ** 2)[:-1]])
        out = torch.empty(len(orders), dtype=torch.complex128, device=DEV)
        for n in np.unique(orders):
            idx = np.nonzero(orders == n)[0]
            A = torch.from_numpy(flat[off[idx][:, None] + np.arange(n * n)].reshape(len(idx), n, n)).to(DEV)
            out[torch.from_numpy(idx).to(DEV)] = _perms_chunked(A)
        return out
    if kind in ("slos", "tree"):
        U = torch.from_numpy(_haar(case["m"], np.random.RandomState(seed))).to(DEV)
        if kind == "slos":
            return _slos_exact(U, _photons(case), case["coefs"], _herald(case) if case["herald"] else None)
        return [_slos_exact(U, r, False) for r in _loss_inputs(case["m"], case["n"], case["lost"])]
    if kind == "mesh":
        return _mesh_exact(case, seed)
    if kind == "gurvits":
        return _gurvits_exact(case, seed)
    if kind == "train":
        return _train_exact(case, seed)
    return None          # samples are whole numbers; the chain's weights follow its float32 draws
