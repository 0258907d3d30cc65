"""GPU parity of the batched Glynn permanent kernel against the CPU oracle.

Bar (north star): relative error <= 1e-10 against a complex128 CPU oracle; the
oracle here is the long-double Glynn of oracle/pcvl_oracle.c, itself pinned in
tests/test_oracle.py.
"""
import ctypes
import math

import numpy as np
import pytest

import oracle
from perceval_amd.utils.workloads import haar_unitary, submatrix_batch

pytestmark = pytest.mark.gpu

REL_TOL = 1e-10


def _rel(a, b):
    return abs(a - b) / max(abs(b), 1e-300)


def _say(msg):
    print(f"[perm-gpu] {msg}", flush=True)


def _gpu_perms(mats):
    from perceval_amd.permanent import permanents
    _say(f"GPU batch of {len(mats)} (orders {sorted(set(int(np.shape(m)[0]) for m in mats))})")
    out = permanents(mats)
    _say("GPU batch done")
    return out


def _oracle(mats):
    _say(f"oracle batch of {len(mats)}")
    out = oracle.perm_batch(mats, precise=True)
    _say("oracle batch done")
    return out


def test_small_orders_vs_brute(gpu):
    rng = np.random.RandomState(1)
    mats = [rng.randn(n, n) + 1j * rng.randn(n, n) for n in range(0, 9) for _ in range(3)]
    got = _gpu_perms(mats)
    for M, g in zip(mats, got):
        ref = oracle.perm_brute(M) if M.shape[0] <= 7 else oracle.perm(M)
        assert _rel(g, ref) < 1e-12, (M.shape, g, ref)


@pytest.mark.parametrize("lo,hi,count", [(0, 11, 300), (4, 6, 33), (10, 12, 17), (11, 11, 3000), (11, 14, 2500)])
def test_small_and_grouped_items_vs_oracle(gpu, lo, hi, count):
    """Orders around the lines between a thread (to 5), 16 lanes (to 10) and a
    wave per matrix, in one batch, with counts off the 16 matrices of a
    workgroup; and queues of so many small items that waves take them in groups,
    executed twice (the cursor goes back to zero)."""
    import torch
    from perceval_amd.permanent import PermanentPlan, pack
    rng = np.random.RandomState(lo + 100 * hi)
    mats = [rng.randn(n, n) + 1j * rng.randn(n, n) for n in rng.randint(lo, hi + 1, count)]
    orders, flat = pack(mats)
    plan = PermanentPlan(orders)
    d = torch.from_numpy(flat).cuda()
    got = [plan(d).cpu().numpy() for _ in range(2)]
    assert np.array_equal(got[0], got[1])
    ref = oracle.perm_batch(mats, precise=True)
    for g, r, M in zip(got[0], ref, mats):
        assert _rel(g, r) < REL_TOL, (M.shape, g, r)


@pytest.mark.parametrize("n", list(range(9, 25)))
def test_wave_orders_vs_oracle(gpu, n):
    U = haar_unitary(64, seed=100 + n)
    rng = np.random.RandomState(n)
    mats = [U[np.ix_(rng.choice(64, n, replace=False), rng.choice(64, n, replace=False))] for _ in range(2)]
    got = _gpu_perms(mats)
    ref = _oracle(mats)
    for g, r in zip(got, ref):
        assert _rel(g, r) < REL_TOL, (n, g, r)


@pytest.mark.parametrize("variant", [1, 2, 3, 4])
@pytest.mark.parametrize("n", [9, 13, 20, 24])
def test_kernel_variants_vs_oracle(gpu, n, variant):
    import torch
    from perceval_amd.permanent import PermanentPlan, pack
    U = haar_unitary(64, seed=300 + n)
    rng = np.random.RandomState(7 * n)
    mats = [U[np.ix_(rng.choice(64, n, replace=False), rng.choice(64, n, replace=False))] for _ in range(3)]
    orders, flat = pack(mats)
    for chunk in (2, 11):
        plan = PermanentPlan(orders, max_chunk_log2=chunk, variant=variant)
        got = plan(torch.from_numpy(flat).cuda()).cpu().numpy()
        plan.close()
        for g, r in zip(got, _oracle(mats)):
            assert _rel(g, r) < REL_TOL, (n, variant, chunk, g, r)


@pytest.mark.parametrize("n", [9, 10, 19, 24, 25, 26])
def test_block_edges_vs_oracle(gpu, n):
    """Orders at the edges of the two kernels of the wave path (odd and even
    columns, two low rows up to order 24, one above), with one block per lane
    (its sign is the lane's), two, and many; Gaussian entries of uneven column
    scale, so that a pair's products and their updates differ by 10^6."""
    import torch
    from perceval_amd.permanent import PermanentPlan, pack
    rng = np.random.RandomState(900 + n)
    mats = [(rng.randn(n, n) + 1j * rng.randn(n, n)) * 10.0 ** rng.uniform(-3, 3, size=n) for _ in range(2)]
    orders, flat = pack(mats)
    ref = _oracle(mats)
    for chunk in (2, 3, 11):
        plan = PermanentPlan(orders, max_chunk_log2=chunk)
        got = plan(torch.from_numpy(flat).cuda()).cpu().numpy()
        plan.close()
        for g, r in zip(got, ref):
            assert _rel(g, r) < REL_TOL, (n, chunk, g, r)


def test_mixed_batch_config_shape(gpu):
    # Same generator as the batched-permanent workload (n uniform in 12..24 from
    # one 64x64 Haar unitary), 4096 matrices; every matrix of order <= 16 and a
    # seeded sample of the larger ones are checked against the oracle.
    _, orders, mats = submatrix_batch(4096, 12, 24, seed=7)
    got = _gpu_perms(mats)
    small = [i for i, n in enumerate(orders) if n <= 16]
    rng = np.random.RandomState(3)
    large = [i for i, n in enumerate(orders) if n > 16]
    sample = small + sorted(rng.choice(large, size=24, replace=False).tolist())
    ref = _oracle([mats[i] for i in sample])
    errs = [_rel(got[i], r) for i, r in zip(sample, ref)]
    assert max(errs) < REL_TOL, max(errs)


def test_order20_batch_and_replay(gpu):
    import torch
    from perceval_amd.permanent import PermanentPlan, pack
    _, orders, mats = submatrix_batch(512, 20, 20, seed=11)
    o, flat = pack(mats)
    plan = PermanentPlan(o)
    d = torch.from_numpy(flat).cuda()
    a = plan(d).cpu().numpy()
    b = plan(d).cpu().numpy()
    plan.close()
    assert np.array_equal(a.view(np.float64), b.view(np.float64)), "replay is not bit-reproducible"
    ref = _oracle(mats[:16])
    for g, r in zip(a[:16], ref):
        assert _rel(g, r) < REL_TOL


def test_identities_order20(gpu):
    n = 20
    rng = np.random.RandomState(5)
    A = haar_unitary(n, seed=9)
    d1 = np.exp(1j * rng.uniform(0, 2 * np.pi, n)) * rng.uniform(0.5, 1.5, n)
    d2 = np.exp(1j * rng.uniform(0, 2 * np.pi, n)) * rng.uniform(0.5, 1.5, n)
    P = np.eye(n)[rng.permutation(n)]
    Q = np.eye(n)[rng.permutation(n)]
    mats = [np.eye(n, dtype=complex), np.ones((n, n), dtype=complex) / 2, A, A.T, P @ A @ Q,
            np.diag(d1) @ A @ np.diag(d2)]
    got = _gpu_perms(mats)
    assert _rel(got[0], 1.0) < 1e-14
    assert _rel(got[1], math.factorial(n) / 2 ** n) < REL_TOL   # all-ones: maximal cancellation
    assert _rel(got[3], got[2]) < REL_TOL
    assert _rel(got[4], got[2]) < REL_TOL
    assert _rel(got[5], np.prod(d1) * np.prod(d2) * got[2]) < REL_TOL


def test_rejects_order_above_max(gpu):
    from perceval_amd.permanent import PermanentPlan
    with pytest.raises(ValueError):
        PermanentPlan([33])


def test_fp64_probe_counts_and_values(gpu):
    import ctypes
    import torch
    from perceval_amd import _native
    lib = _native.load()
    out = torch.empty(4 * 256, dtype=torch.float64, device="cuda")
    flops = ctypes.c_int64()
    _native.check(lib.pcvl_probe_fp64_fma(4, 10, _native.ptr(out), ctypes.byref(flops), _native.stream_handle()),
                  "probe")
    assert flops.value == 4 * 256 * 16 * 10 * 2
    got = out.cpu().numpy()
    a, b = 0.999999999, 1e-9
    for lane in (0, 1, 255, 300):
        ref = 0.0
        for k in range(16):
            c = float((lane % 256) + k)
            for _ in range(10):
                c = c * a + b
            ref += c
        assert abs(got[lane] - ref) <= 1e-12 * abs(ref)
    with pytest.raises(ValueError):
        _native.check(lib.pcvl_probe_fp64_fma(0, 10, _native.ptr(out), ctypes.byref(flops), None), "probe")


def test_plan_refuses_more_work_items_than_it_can_index(gpu):
    """4096 order-28 matrices cut into 2^2-step chunks need 2^31 work items:
    the plan returns the range status instead of overflowing its 32-bit
    partial-sum slots."""
    from perceval_amd._native import NativeError
    from perceval_amd.permanent import PermanentPlan
    with pytest.raises(NativeError, match="work items"):
        PermanentPlan([28] * 4096, max_chunk_log2=2)
    PermanentPlan([28] * 4, max_chunk_log2=11).close()


@pytest.mark.parametrize("n", [11, 12])
@pytest.mark.parametrize("variant", [0, 2])
def test_smallest_orders_of_the_wave_path(gpu, n, variant):
    """The smallest orders that take waves: one block per lane (its sign is the
    lane's), two, and as many as fit, with two low rows and with one."""
    import torch
    from perceval_amd.permanent import PermanentPlan, pack
    rng = np.random.RandomState(n)
    mats = [(rng.randn(n, n) + 1j * rng.randn(n, n)) * 10.0 ** rng.uniform(-3, 3, size=n) for _ in range(5)]
    orders, flat = pack(mats)
    ref = _oracle(mats)
    for chunk in (2, 3, 11):
        plan = PermanentPlan(orders, max_chunk_log2=chunk, variant=variant)
        got = plan(torch.from_numpy(flat).cuda()).cpu().numpy()
        plan.close()
        for g, r in zip(got, ref):
            assert _rel(g, r) < REL_TOL, (n, chunk, variant, g, r)


def test_small_matrices_in_several_launches(gpu):
    """More matrices of 16 lanes each than one launch takes (2^22), behind some
    of a thread each: all of them share a few matrices."""
    import torch
    from perceval_amd import _native
    from perceval_amd.permanent import pack
    lib = _native.load()
    rng = np.random.RandomState(3)
    mats = [rng.randn(n, n) + 1j * rng.randn(n, n) for n in (3, 6, 7)]
    orders, flat = pack(mats)
    offs = np.concatenate([[0], np.cumsum(orders.astype(np.int64) ** 2)[:-1]])
    which = np.arange((1 << 22) + 5000) % 2 + 1
    which[::1000] = 0
    ns = np.ascontiguousarray(orders[which], dtype=np.int32)
    of = np.ascontiguousarray(offs[which], dtype=np.int64)
    out = torch.full((len(which),), complex(np.nan, np.nan), dtype=torch.complex128, device="cuda")
    d = torch.from_numpy(flat).cuda()
    assert lib.pcvl_perm_batch(_native.ptr(d), ns.ctypes.data_as(ctypes.POINTER(ctypes.c_int32)),
                               of.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)), len(ns), _native.ptr(out),
                               _native.stream_handle()) == 0
    ref = oracle.perm_batch(mats, precise=True)
    got = out.cpu().numpy()
    for k, r in enumerate(ref):
        assert np.max(np.abs(got[which == k] - r)) < REL_TOL * abs(r), k
