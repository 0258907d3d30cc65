"""Learned Metropolis independence sampler: the proposal network's kernels
against the NumPy oracle (oracle/mlp.py), exactness of q and p, the chain scan
against a host restatement, and the sampler's output law against exact
distributions and plain Clifford-Clifford samples."""
import math
from collections import Counter

import numpy as np
import pytest

import oracle
from oracle import mlp as mlp_oracle
from perceval_amd.utils.workloads import haar_unitary

pytestmark = pytest.mark.gpu


def _say(msg):
    print(f"[mis-gpu] {msg}", flush=True)


def _seqs_from_cc(U, inp, count, seed):
    s = oracle.cc_samples(U, inp, count, seed=seed)
    return np.array([[j for j, v in enumerate(row) for _ in range(v)] for row in s], dtype=np.int32)


def test_network_gradients_vs_oracle(gpu):
    import torch
    from perceval_amd.mis import ProposalNet
    m, n = 10, 4
    U = haar_unitary(m, seed=2)
    seqs = _seqs_from_cc(U, [1] * n + [0] * (m - n), 64, seed=1)
    net = ProposalNet(m, n, hidden=32, seed=3)
    # non-trivial biases and second-layer weights
    g = torch.Generator().manual_seed(5)
    net.b1.copy_(torch.randn(32, generator=g).float().cuda() * 0.1)
    net.W2.copy_(torch.randn(m, 32, generator=g).float().cuda() * 0.3)
    net.b2.copy_(torch.randn(m, generator=g).float().cuda() * 0.1)
    net.refresh_bf16()
    d = torch.from_numpy(seqs).cuda()
    x, lo, tgt = net.teacher_forcing(d)
    loss, grads = net.loss_and_grads(x, lo, tgt, 1.0 / 64)
    X, LO, TG = mlp_oracle.features(seqs, m)
    assert np.array_equal(x.cpu().numpy(), X) and np.array_equal(lo.cpu().numpy(), LO)
    ref_loss, ref_grads = mlp_oracle.loss_and_grads(*(p.double().cpu().numpy() for p in net.params), X, LO, TG,
                                                    1.0 / 64)
    assert np.allclose(loss.cpu().numpy(), ref_loss, rtol=1e-5, atol=1e-5)
    for gg, rg in zip(grads, ref_grads):
        gg = gg.double().cpu().numpy()
        assert np.max(np.abs(gg - rg)) <= 1e-5 * max(1.0, np.max(np.abs(rg))), np.max(np.abs(gg - rg))


@pytest.mark.parametrize("m,n,H,B", [(1, 1, 1, 1), (3, 2, 40, 17), (17, 15, 33, 70), (33, 16, 64, 3),
                                     (60, 20, 256, 700), (64, 32, 256, 300), (64, 33, 256, 20), (65, 3, 16, 50),
                                     (10, 4, 257, 50)])
def test_training_step_shapes_vs_oracle(gpu, m, n, H, B):
    """Loss, gradients and the Adam step on both sides of the one-launch pass
    (64 modes, 96 inputs, 256 hidden units): one row to several tiles of 32 per
    workgroup, widths around multiples of 16, rows without an allowed target.
    The bars are those of the gradient and Adam tests above and below."""
    import torch
    from perceval_amd.mis import ProposalNet
    rng = np.random.RandomState(m + n)
    seqs = np.sort(rng.randint(0, m, size=(B, n)), axis=1).astype(np.int32)
    net = ProposalNet(m, n, hidden=H, seed=3)
    for p, sd in zip(net.params, (0.3, 0.1, 0.3, 0.1)):
        p.copy_(torch.from_numpy((sd * rng.randn(*p.shape)).astype(np.float32)).cuda())
    net.refresh_bf16()
    x, lo, tgt = net.teacher_forcing(torch.from_numpy(seqs).cuda())
    X, LO, TG = mlp_oracle.features(seqs, m)
    assert np.array_equal(x.cpu().numpy(), X) and np.array_equal(lo.cpu().numpy(), LO)
    assert np.array_equal(tgt.cpu().numpy(), TG)
    bad = np.arange(0, B * n, 7) if B * n > 7 else np.arange(0)
    tgt[torch.from_numpy(bad).cuda()] = torch.from_numpy(np.where(bad % 2, m, -1).astype(np.int32)).cuda()
    w0 = [p.double().cpu().numpy() for p in net.params]
    loss, grads = net.loss_and_grads(x, lo, tgt, 1.0 / B)
    loss2, grads2 = net.loss_and_grads(x, lo, tgt, 1.0 / B)
    assert torch.equal(loss, loss2) and all(torch.equal(a, b) for a, b in zip(grads, grads2))
    keep = np.setdiff1d(np.arange(B * n), bad)
    ref_loss, ref_grads = mlp_oracle.loss_and_grads(*w0, X[keep], LO[keep], TG[keep], 1.0 / B)
    got = loss.cpu().numpy()
    assert np.isposinf(got[bad]).all()
    assert np.allclose(got[keep], ref_loss, rtol=1e-5, atol=1e-5)
    for gg, rg in zip(grads, ref_grads):
        gg = gg.double().cpu().numpy()
        assert np.max(np.abs(gg - rg)) <= 1e-5 * max(1.0, np.max(np.abs(rg))), np.max(np.abs(gg - rg))
    net.adam_step(grads, lr=1e-2)
    for p, w, gg in zip(net.params, w0, grads):
        ref, _, _ = mlp_oracle.adam(w, gg.double().cpu().numpy(), np.zeros(w.shape), np.zeros(w.shape), 1e-2, 0.9,
                                    0.999, 1e-8, 1)
        assert np.allclose(p.cpu().numpy(), ref, rtol=1e-5, atol=1e-6)
    assert torch.equal(net.W1b, net.W1.bfloat16()) and torch.equal(net.W2b, net.W2.bfloat16())


def test_adam_step_vs_oracle(gpu):
    import torch
    from perceval_amd import _native
    lib = _native.load()
    rng = np.random.RandomState(0)
    w = rng.randn(1000).astype(np.float32)
    g = rng.randn(1000).astype(np.float32)
    dw, dg = torch.from_numpy(w).cuda(), torch.from_numpy(g).cuda()
    m1, m2 = torch.zeros_like(dw), torch.zeros_like(dw)
    wb = torch.empty(1000, dtype=torch.bfloat16, device="cuda")
    rw, rm1, rm2 = w.astype(np.float64), np.zeros(1000), np.zeros(1000)
    for step in (1, 2, 3):
        _native.check(lib.pcvl_mlp_adam(_native.ptr(dw), _native.ptr(dg), _native.ptr(m1), _native.ptr(m2),
                                        _native.ptr(wb), 1000, 1e-2, 0.9, 0.999, 1e-8, step,
                                        _native.stream_handle()), "adam")
        rw, rm1, rm2 = mlp_oracle.adam(rw, g.astype(np.float64), rm1, rm2, 1e-2, 0.9, 0.999, 1e-8, step)
    assert np.allclose(dw.cpu().numpy(), rw, rtol=1e-5, atol=1e-6)
    assert np.array_equal(wb.float().cpu().numpy(), mlp_oracle.bf16_round(dw.cpu().numpy()).astype(np.float32))


@pytest.mark.parametrize("R,Mo,No", [(1, 3, 5), (257, 60, 256), (40960, 256, 80), (1000, 70, 0)])
def test_wgrad_and_colsum_vs_numpy(gpu, R, Mo, No):
    import ctypes
    import torch
    from perceval_amd import _native
    lib = _native.load()
    rng = np.random.RandomState(R + Mo)
    dY = rng.randn(R, Mo).astype(np.float32)
    X = rng.randn(R, max(No, 1)).astype(np.float32)[:, :No].copy()
    f = ctypes.c_int64()
    _native.check(lib.pcvl_mlp_wgrad_workspace(R, Mo, No, ctypes.byref(f)), "ws")
    work = torch.empty(f.value, dtype=torch.float32, device="cuda")
    d_dY, d_X = torch.from_numpy(dY).cuda(), torch.from_numpy(X).cuda()
    dW = torch.empty((Mo, No), dtype=torch.float32, device="cuda")
    db = torch.empty(Mo, dtype=torch.float32, device="cuda")
    for _ in range(2):   # deterministic: the same bits twice
        _native.check(lib.pcvl_mlp_wgrad(_native.ptr(d_dY), Mo, _native.ptr(d_X) if No else None, max(No, 1), R, Mo,
                                         No, _native.ptr(dW) if No else None, _native.ptr(db), _native.ptr(work),
                                         work.numel(), _native.stream_handle()), "wgrad")
        got = (dW.cpu().numpy().copy(), db.cpu().numpy().copy())
        if _ == 0:
            first = got
    assert np.array_equal(first[0], got[0]) and np.array_equal(first[1], got[1])
    ref_W = dY.astype(np.float64).T @ X.astype(np.float64)
    ref_b = dY.astype(np.float64).sum(axis=0)
    scale = np.sqrt(R)
    assert np.max(np.abs(got[0] - ref_W), initial=0.0) <= 1e-5 * scale
    assert np.max(np.abs(got[1] - ref_b)) <= 1e-5 * scale
    cs = torch.empty(Mo, dtype=torch.float32, device="cuda")
    _native.check(lib.pcvl_mlp_colsum(_native.ptr(d_dY), R, Mo, _native.ptr(cs), _native.stream_handle()), "colsum")
    assert np.max(np.abs(cs.cpu().numpy() - ref_b)) <= 1e-5 * scale
    with pytest.raises(ValueError):
        lib_rc = lib.pcvl_mlp_wgrad(_native.ptr(d_dY), Mo, _native.ptr(d_X), max(No, 1), R, Mo, No, None,
                                    _native.ptr(db), _native.ptr(work), 0, _native.stream_handle())
        _native.check(lib_rc, "wgrad small workspace")


def test_sampling_gives_exact_log_q(gpu):
    from perceval_amd.mis import ProposalNet
    m, n = 12, 5
    net = ProposalNet(m, n, hidden=64, seed=1)
    seq, logq = net.sample(512, seed=9)
    s = seq.cpu().numpy()
    assert (np.diff(s, axis=1) >= 0).all() and s.min() >= 0 and s.max() < m
    assert np.allclose(logq.cpu().numpy(), net.log_q(seq).cpu().numpy(), atol=2e-4)
    # q sums to one over the whole space (m=12, n=5: 4368 states)
    import torch
    states = oracle.fock_enumerate(m, n)
    seqs = np.array([[j for j, v in enumerate(r) for _ in range(v)] for r in states], dtype=np.int32)
    tot = torch.exp(net.log_q(torch.from_numpy(seqs).cuda())).sum().item()
    assert abs(tot - 1.0) < 1e-4


def test_fused_sampler_matches_stepwise_and_its_own_q(gpu):
    """The one-launch sampler draws with the same uniforms as the stepwise
    path, so the draws coincide except where fp32 rounding of the two
    evaluation orders moves a CDF boundary; its log q is exact for what it drew
    and its empirical law matches q."""
    import torch
    from perceval_amd.mis import ProposalNet
    m, n = 12, 5
    net = ProposalNet(m, n, hidden=64, seed=4)
    g = torch.Generator().manual_seed(2)
    net.b1.copy_(torch.randn(64, generator=g).float().cuda() * 0.2)
    net.b2.copy_(torch.randn(m, generator=g).float().cuda() * 0.5)
    net.W2.mul_(8.0)
    net.refresh_bf16()
    assert net.fused_ok()
    sf, qf = net.sample(4096, seed=21, first=7)
    ss, qs = net.sample(4096, seed=21, first=7, fused=False)
    same = (sf == ss).all(dim=1)
    assert same.float().mean().item() > 0.99
    assert torch.allclose(qf[same], qs[same], atol=1e-4)
    assert torch.allclose(qf, net.log_q(sf), atol=2e-4)
    # empirical law of 200k fused draws against q over the whole space (m=6, n=3: 56 states)
    m2, n2 = 6, 3
    net2 = ProposalNet(m2, n2, hidden=32, seed=5)
    net2.W2.mul_(10.0)
    net2.refresh_bf16()
    seqs, _ = net2.sample(200000, seed=3)
    states = oracle.fock_enumerate(m2, n2)
    allseq = np.array([[j for j, v in enumerate(r) for _ in range(v)] for r in states], dtype=np.int32)
    q = torch.exp(net2.log_q(torch.from_numpy(allseq).cuda())).cpu().numpy()
    assert abs(q.sum() - 1.0) < 1e-4
    key = {tuple(r): i for i, r in enumerate(allseq.tolist())}
    cnt = np.zeros(len(allseq))
    for r in seqs.cpu().numpy().tolist():
        cnt[key[tuple(r)]] += 1
    tvd = 0.5 * np.abs(cnt / cnt.sum() - q).sum()
    _say(f"fused sampler TVD to q: {tvd:.4f}")
    assert tvd < 0.01


def test_log_p_vs_oracle(gpu):
    import torch
    from perceval_amd.mis import LearnedMIS, ProposalNet
    m, n = 12, 5
    U = haar_unitary(m, seed=4)
    inp = [1] * n + [0] * (m - n)
    net = ProposalNet(m, n, hidden=16)
    mis = LearnedMIS(U, inp, net, chunk=256)
    states = oracle.fock_enumerate(m, n)[::17]
    seqs = np.array([[j for j, v in enumerate(r) for _ in range(v)] for r in states], dtype=np.int32)
    lp = mis.log_p(torch.from_numpy(seqs).cuda()).cpu().numpy()
    for s, v in zip(states, lp):
        ref = abs(oracle.perm(oracle.submatrix(U, inp, s))) ** 2 / oracle.prodnfact(s)
        assert abs(math.exp(v) - ref) <= 1e-12 + 1e-10 * ref
    mis.close()


@pytest.mark.parametrize("m,n", [(6, 5), (12, 8), (60, 20)])
def test_multiset_permanents_vs_oracle(gpu, m, n):
    import torch
    from perceval_amd.mis import LearnedMIS, ProposalNet
    U = haar_unitary(m, seed=m + n)
    inp = [1] * n + [0] * (m - n)
    rng = np.random.RandomState(n)
    # sequences with many collisions, a few without, and all photons in one mode
    seqs = [np.sort(rng.randint(0, max(2, m // 3), size=n)) for _ in range(12)]
    seqs += [np.sort(rng.choice(m, n, replace=False)) for _ in range(3)]
    seqs += [np.full(n, m - 1), np.array([0] * (n // 2) + [1] * (n - n // 2))]
    seqs = np.array(seqs, dtype=np.int32)
    mis = LearnedMIS(U, inp, ProposalNet(m, n, hidden=8), chunk=64)
    got = mis.permanents(torch.from_numpy(seqs).cuda()).cpu().numpy()
    for s, g in zip(seqs, got):
        occ = np.bincount(s, minlength=m)
        ref = oracle.perm(oracle.submatrix(U, inp, occ))
        assert abs(g - ref) <= 1e-10 * abs(ref) + 1e-14, (s, g, ref)
    mis.close()


@pytest.mark.parametrize("n", [5, 6, 7, 24, 25])
def test_multiset_permanents_block_edges(gpu, n):
    """Orders around the block loop's limits (none below 6, two low rows up to
    24, one above), with 0..4 unique rows besides the fixed one: fewer than
    the low rows, exactly them (one block, no flip), and one flip more."""
    import torch
    from perceval_amd.mis import LearnedMIS, ProposalNet
    m = 30
    U = haar_unitary(m, seed=50 + n)
    inp = [1] * n + [0] * (m - n)
    seqs = []
    for unique in range(0, min(n, 6)):
        left = n - unique
        if left == 1:
            continue
        pair = left - 2 if left > 3 else left     # groups of left - 2 and 2, or one of left
        s = list(range(10, 10 + unique)) + [3] * pair + [7] * (left - pair)
        seqs.append(sorted(s))
    seqs = np.array(seqs, dtype=np.int32)
    mis = LearnedMIS(U, inp, ProposalNet(m, n, hidden=8), chunk=64)
    got = mis.permanents(torch.from_numpy(seqs).cuda()).cpu().numpy()
    for s, g in zip(seqs, got):
        ref = oracle.perm_large(oracle.submatrix(U, inp, np.bincount(s, minlength=m)), threads=8)
        assert abs(g - ref) <= 1e-10 * abs(ref) + 1e-14, (s, g, ref)
    mis.close()


def test_multiset_permanents_mixed_costs_deterministic(gpu):
    """A batch mixing collision-free, bunched and single-mode proposals (costs
    from 1 to 2^15 terms), against the oracle, and bit-identical when run twice."""
    import torch
    from perceval_amd.mis import LearnedMIS, ProposalNet
    m, n = 40, 16
    U = haar_unitary(m, seed=5)
    inp = [1] * n + [0] * (m - n)
    rng = np.random.RandomState(1)
    seqs = []
    for k in range(300):
        kind = k % 4
        if kind == 0:
            seqs.append(np.sort(rng.choice(m, n, replace=False)))
        elif kind == 1:
            seqs.append(np.sort(rng.randint(0, m, size=n)))
        elif kind == 2:
            seqs.append(np.sort(rng.randint(0, 4, size=n)))
        else:
            seqs.append(np.full(n, rng.randint(m)))
    seqs = np.array(seqs, dtype=np.int32)
    mis = LearnedMIS(U, inp, ProposalNet(m, n, hidden=8), chunk=512)
    d = torch.from_numpy(seqs).cuda()
    a = mis.permanents(d).cpu().numpy()
    b = mis.permanents(d).cpu().numpy()
    assert np.array_equal(a, b)
    for s_, g in list(zip(seqs, a))[::7]:
        ref = oracle.perm(oracle.submatrix(U, inp, np.bincount(s_, minlength=m)))
        assert abs(g - ref) <= 1e-10 * abs(ref) + 1e-14, (s_, g, ref)
    mis.close()


@pytest.mark.parametrize("B", [1, 37, 64, 5000])
def test_chain_scan_vs_host_restatement(gpu, B):
    import torch
    from perceval_amd import _native
    lib = _native.load()
    rng = np.random.RandomState(3)
    logw = rng.randn(B) * 2
    d = torch.from_numpy(logw).cuda()
    state = torch.empty(B, dtype=torch.int64, device="cuda")
    acc = torch.zeros(1, dtype=torch.int64, device="cuda")
    _native.check(lib.pcvl_mis_chain(_native.ptr(d), B, 0.3, 77, 10, _native.ptr(state), _native.ptr(acc),
                                     _native.stream_handle()), "chain")
    cur, idx, ref, nacc = 0.3, -1, [], 0
    for t in range(B):
        dlt = logw[t] - cur
        if dlt >= 0 or math.log(oracle.uniform(77, 10 + t, 0)) < dlt:
            cur, idx, nacc = logw[t], t, nacc + 1
        ref.append(idx)
    assert np.array_equal(state.cpu().numpy(), np.array(ref)) and acc.item() == nacc


@pytest.mark.parametrize("first", [0, 1000])
def test_run_vs_host_replay(gpu, first):
    """A whole run: the chain over the proposals it returns, started from
    x0's own weight, replayed on the host with the oracle's uniforms."""
    import torch
    from perceval_amd.mis import LearnedMIS, ProposalNet
    m, n = 8, 3
    U = haar_unitary(m, seed=12)
    inp = [1, 1, 1] + [0] * (m - 3)
    net = ProposalNet(m, n, hidden=32, seed=5)
    net.train(torch.from_numpy(_seqs_from_cc(U, inp, 4000, seed=6)).cuda(), epochs=1, batch=1024)
    mis = LearnedMIS(U, inp, net, chunk=1024)
    x0 = torch.from_numpy(_seqs_from_cc(U, inp, 1, seed=9)[0]).cuda()
    count, seed = 3000, 21
    res = mis.run(count, seed=seed, x0_seq=x0, first=first)
    props = res["proposals"].cpu().numpy()
    logw = res["logw"].cpu().numpy()
    # the proposals' weights against a separate scoring (their log q comes
    # from the sampler's own fp32 logits, equal to net.log_q up to rounding)
    lp = mis.log_p(res["proposals"]).cpu().numpy()
    lq = net.log_q(res["proposals"]).cpu().numpy()
    assert np.allclose(logw, lp - lq, rtol=0, atol=1e-3)
    x0s = x0.reshape(1, n).to(torch.int32)
    cur = float((mis.log_p(x0s) - net.log_q(x0s))[0].item())
    held, nacc, ref = x0.cpu().numpy(), 0, []
    for t in range(count):
        dlt = logw[t] - cur
        if dlt >= 0 or math.log(oracle.uniform(seed ^ 0x5DEECE66D, first + t, 0)) < dlt:
            cur, held, nacc = logw[t], props[t], nacc + 1
        ref.append(held)
    assert np.array_equal(res["seq"].cpu().numpy(), np.array(ref))
    assert res["acceptance"] == nacc / count
    mis.close()


@pytest.mark.parametrize("trained", [False, True])
def test_chain_law_small(gpu, trained):
    import torch
    from perceval_amd.mis import LearnedMIS, ProposalNet, seq_to_occ
    m, n = 5, 3
    U = haar_unitary(m, seed=31)
    inp = [1, 1, 1, 0, 0]
    net = ProposalNet(m, n, hidden=32, seed=2)
    if trained:
        net.train(torch.from_numpy(_seqs_from_cc(U, inp, 20000, seed=4)).cuda(), epochs=3, batch=1024)
    mis = LearnedMIS(U, inp, net, chunk=4096)
    x0 = torch.from_numpy(_seqs_from_cc(U, inp, 1, seed=8)[0]).cuda()
    res = mis.run(60000, seed=5, x0_seq=x0)
    occ = seq_to_occ(res["seq"], m).cpu().numpy()
    exact = oracle.distribution_exact(U, inp)
    c = Counter(map(tuple, occ.tolist()))
    tvd = 0.5 * sum(abs(c.get(s, 0) / len(occ) - p) for s, p in exact.items())
    _say(f"trained={trained} acceptance={res['acceptance']:.3f} tvd={tvd:.4f}")
    assert tvd < 0.02
    mis.close()


def test_learned_proposal_beats_untrained_m20_n6(gpu):
    import torch
    from perceval_amd.mis import LearnedMIS, ProposalNet, marginal_tvds, seq_to_occ
    from perceval_amd.sampling import cc_samples
    m, n = 20, 6
    U = haar_unitary(m, seed=77)
    inp = [1] * n + [0] * (m - n)
    train = cc_samples(U, inp, 30000, seed=1)
    ref = cc_samples(U, inp, 30000, seed=2)
    from perceval_amd.mis import occ_to_seq
    tseq = occ_to_seq(torch.from_numpy(train).cuda(), n)
    x0 = tseq[0]
    accs = {}
    for trained in (False, True):
        net = ProposalNet(m, n, hidden=128, seed=0)
        if trained:
            hist = net.train(tseq, epochs=4, batch=2048)
            _say(f"train nll {hist}")
        mis = LearnedMIS(U, inp, net, chunk=8192)
        res = mis.run(30000, seed=11, x0_seq=x0)
        occ = seq_to_occ(res["seq"], m).cpu().numpy()
        tv = marginal_tvds(occ, ref)
        accs[trained] = res["acceptance"]
        _say(f"trained={trained} acceptance={res['acceptance']:.3f} {tv}")
        mis.close()
        if trained:
            assert tv["tvd1_mean"] < 0.02
    assert accs[True] > accs[False]


def test_multiset_permanents_many_short_slices(gpu):
    """So many short slices that waves take several at a time: bunched proposals
    of 16 photons in 12 modes, against the plain permanents of the submatrices."""
    import torch
    from perceval_amd.mis import LearnedMIS, ProposalNet
    m, n, B = 12, 16, 60000
    U = haar_unitary(m, seed=6)
    inp = [2] * 4 + [1] * 8
    rng = np.random.RandomState(4)
    seqs = torch.from_numpy(np.sort(rng.randint(0, m, size=(B, n)), axis=1).astype(np.int32)).cuda()
    net = ProposalNet(m, n, hidden=8)
    a = LearnedMIS(U, inp, net, chunk=B).permanents(seqs).cpu().numpy()
    b = LearnedMIS(U, inp, net, chunk=B, multiset=False).permanents(seqs).cpu().numpy()
    # both sum 2^15 terms of products of 16 column sums in double: 1e-12 of the
    # largest permanent of the batch
    assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(b))


def test_training_step_without_a_gradient_or_photons(gpu):
    """A missing gradient is refused before a kernel reads it; a network of no
    photons takes the general products."""
    import torch
    from perceval_amd.mis import ProposalNet
    net = ProposalNet(6, 3, hidden=16)
    before = [p.clone() for p in net.params]
    grads = [torch.ones_like(p) for p in net.params]
    with pytest.raises(AttributeError):
        net.adam_step(grads[:1] + [None] + grads[2:])
    assert all(torch.equal(a, b) for a, b in zip(before, net.params))
    net.adam_step(grads[:2])
    assert not torch.equal(before[1], net.params[1]) and torch.equal(before[2], net.params[2])
    empty = ProposalNet(4, 0, hidden=8)
    x = torch.zeros((3, 4), dtype=torch.float32, device="cuda")
    lo = torch.zeros(3, dtype=torch.int32, device="cuda")
    loss, grads = empty.loss_and_grads(x, lo, lo, 1.0)
    assert torch.allclose(loss, torch.full_like(loss, np.log(4.0)), atol=1e-6) and grads[0].shape == (8, 4)
