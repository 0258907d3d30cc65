"""GPU Gurvits estimates (NaiveApprox) against the oracle restatement (same
counter-based samples, so the means agree to rounding), exact cases, the 99%
coverage of the error bound, and the NaiveApprox backend API."""
import numpy as np
import pytest

import oracle
from perceval_amd.utils.workloads import haar_unitary

pytestmark = pytest.mark.gpu


def _say(msg):
    print(f"[gurvits-gpu] {msg}", flush=True)


@pytest.mark.parametrize("orders", [[0, 1, 2, 3], [5, 8, 12], [16, 20, 24], [30, 31, 32], [40, 48]])
def test_gurvits_batch_vs_oracle(gpu, orders):
    from perceval_amd.permanent import gurvits
    U = haar_unitary(64, seed=sum(orders) + 1)
    rng = np.random.RandomState(len(orders))
    mats = [U[np.ix_(rng.choice(64, n, replace=False), rng.choice(64, n, replace=False))] * 2.0 for n in orders]
    iters, seed, stream0 = 3000, 99, 5
    est, err = gurvits(mats, iters, seed=seed, stream0=stream0)
    _say(f"orders {orders}")
    for b, M in enumerate(mats):
        ref_est, ref_err = oracle.gurvits(M, iters, seed=seed, stream=stream0 + b)
        scale = max(ref_err * np.sqrt(iters) / 2.5758293035489004, abs(ref_est), 1e-300)
        assert abs(est[b] - ref_est) <= 1e-11 * scale, (orders[b], est[b], ref_est)
        # the bound comes from E|X|^2 - |mean|^2, whose rounding (summation
        # order) matters only when the variance is at rounding level
        assert abs(err[b] - ref_err) <= 1e-6 * ref_err + 1e-6 * scale / np.sqrt(iters), (orders[b], err[b], ref_err)


@pytest.mark.parametrize("orders", [[9, 15, 16], [3, 17, 31, 32], [30, 30]])
def test_gurvits_integer_products_vs_oracle(gpu, orders):
    """Calls long enough for the integer products: padding rows and none, an
    order below the kernel's, entries at the ends of the fixed point (rows of
    scale 2^-300 and 2^200, zero rows and components, powers of two), and
    matrices whose entries keep the FP64 products (a component of 2^-50 of its
    row's largest; one that is not finite) beside ones that do not.  Sums are
    compared as in test_gurvits_batch_vs_oracle."""
    from perceval_amd.permanent import gurvits
    rng = np.random.RandomState(sum(orders))
    mats = [(rng.randn(n, n) + 1j * rng.randn(n, n)) / np.sqrt(n) for n in orders]
    n = orders[-1]
    scaled = (rng.randn(n, n) + 1j * rng.randn(n, n)) / np.sqrt(n)
    scaled[0] *= 2.0 ** -300
    scaled[1] *= 2.0 ** 200
    structured = rng.randint(-1, 2, size=(n, n)) * 2.0 ** rng.randint(-9, 1, size=(n, n)) + 0j
    structured[:, 1] = 1j
    tiny = mats[-1].copy()
    tiny[2, 3] = 2.0 ** -50
    zero_row = mats[-1].copy()
    zero_row[n - 1] = 0.0
    nan = mats[-1].copy()
    nan[0, 0] = np.nan
    mats += [scaled, structured, tiny, zero_row, nan]
    iters, seed = (1 << 22) // len(mats) + 77, 7
    est, err = gurvits(mats, iters, seed=seed)
    assert np.isnan(est[-1]) and est[-2] == 0.0 and err[-2] == 0.0
    for b, M in enumerate(mats[:-2]):
        ref_est, ref_err = oracle.gurvits(M, iters, seed=seed, stream=b)
        scale = max(ref_err * np.sqrt(iters) / 2.5758293035489004, abs(ref_est), 1e-300)
        assert abs(est[b] - ref_est) <= 1e-11 * scale, (b, est[b], ref_est)
        assert abs(err[b] - ref_err) <= 1e-6 * ref_err, (b, err[b], ref_err)


def test_gurvits_exact_cases(gpu):
    from perceval_amd.permanent import gurvits
    est, err = gurvits([np.eye(7), np.array([[3 - 2j]]), np.zeros((0, 0))], 100, seed=3)
    assert est[0] == 1.0 and est[1] == 3 - 2j and est[2] == 1.0


def test_gurvits_coverage_and_convergence(gpu):
    from perceval_amd.permanent import gurvits
    U = haar_unitary(12, seed=4)
    A = U[:8, :8]
    exact = oracle.perm(A)
    est, err = gurvits([A] * 256, 4000, seed=11)
    misses = int(np.sum(np.abs(est - exact) > err))
    _say(f"coverage misses {misses} / 256")
    assert misses <= 10
    big, berr = gurvits([A], 4_000_000, seed=12)
    assert abs(big[0] - exact) <= berr[0] and berr[0] < 0.1 * np.mean(err)


def test_naive_approx_backend(gpu):
    from perceval_amd.backends import BackendFactory
    from perceval_amd.components import BS, Unitary
    from perceval_amd.utils.states import BasicState
    from perceval_amd.components import Circuit
    # the reference wiring test: identity circuit on one mode
    b = BackendFactory.get_backend("NaiveApprox")
    b.set_circuit(Circuit(1))
    b.set_input_state(BasicState([1]))
    assert b.all_prob() == [1.0]
    assert b.probability(BasicState([1])) == 1.0
    # confidence intervals contain the exact probabilities (8 modes, 4 photons)
    U = haar_unitary(8, seed=21)
    approx = BackendFactory.get_backend("NaiveApprox", gurvits_iterations=200000)
    exact = BackendFactory.get_backend("Naive")
    for be in (approx, exact):
        be.set_circuit(Unitary(U))
        be.set_input_state(BasicState([1, 1, 1, 1, 0, 0, 0, 0]))
    # one estimate per output; each is a 99% statement (coverage itself is
    # tested over 256 trials above), so the truth is checked at 1.5x the bound
    for out in ([1, 1, 1, 1, 0, 0, 0, 0], [0, 0, 0, 0, 1, 1, 1, 1], [2, 0, 1, 0, 0, 1, 0, 0], [4, 0, 0, 0, 0, 0, 0, 0]):
        ref = exact.prob_amplitude(BasicState(out))
        a, e = approx.prob_amplitude_with_error(BasicState(out))
        assert abs(a - ref) <= 1.5 * e, (out, a, ref, e)
        lo, hi = approx.probability_confidence_interval(BasicState(out))
        assert 0.0 <= lo <= hi <= 1.0 and hi - lo > 0.0
    # photon-number mismatch: amplitude 0 with no error
    assert approx.prob_amplitude_with_error(BasicState([1, 0, 0, 0, 0, 0, 0, 0])) == (0j, 0.0)
    probs = np.array(approx.all_prob())
    assert len(probs) == 330 and abs(probs.sum() - 1.0) < 0.05
    assert approx.name == "NaiveApprox"
    _ = BS  # noqa: F841


def _draws(seed, stream, iters):
    """Signs' bits of the samples 0..iters-1 of a stream (the counter-based
    generator of the kernels)."""
    def mix(x):
        x = x + np.uint64(0x9E3779B97F4A7C15)
        x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return x ^ (x >> np.uint64(31))
    with np.errstate(over="ignore"):
        key = mix(np.uint64(seed) ^ mix(np.uint64(stream)))
        return mix(key + np.arange(iters, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15))


@pytest.mark.parametrize("n", [10, 16, 21, 32])
def test_gurvits_cancelling_rows_are_exact(gpu, n):
    """Rows whose large entries cancel before weak couplings are added: two rows
    (a, a, w...) and (a, -a, w...) leave the sum of the weak ones in every draw.
    Every operand is held in full, so the mean is within 4 n roundings of the
    terms (a row sum's last bits and a complex product each) and the 100 of the
    longest chain of additions of terms from the long double
    mean over the same draws, whether a matrix takes the integer products
    (couplings down to 2^-24 of the pair) or the FP64 ones (below)."""
    from perceval_amd.permanent import gurvits
    rng = np.random.RandomState(n)
    powers = (12, 20, 23, 27, 36)
    mats = []
    for k in powers:
        M = (rng.randn(n, n) + 1j * rng.randn(n, n)) / np.sqrt(n)
        phase = np.exp(2j * np.pi * rng.rand(2, n)) * (1.0 + rng.rand(2, n))
        M[:2] = phase * 2.0 ** -k
        M[0, :2] = rng.randn() + 1j * rng.randn()
        M[1, :2] = M[0, 0], -M[0, 0]
        mats.append(M)
    iters, seed = (1 << 16) + 5, 3
    est, _ = gurvits(mats + [mats[0]] * 59, iters, seed=seed)   # long enough for the integer products
    for b, (k, M) in enumerate(zip(powers, mats)):
        bits = _draws(seed, b, iters)
        tot, size = np.clongdouble(0), np.longdouble(0)
        A = M.astype(np.clongdouble)
        for s0 in range(0, iters, 1 << 16):
            part = bits[s0:s0 + (1 << 16)]
            x = 1 - 2 * ((part[:, None] >> np.arange(n, dtype=np.uint64)) & np.uint64(1)).astype(np.longdouble)
            term = x.prod(axis=1).astype(np.clongdouble)
            for i in range(n):
                y = np.zeros(len(part), dtype=np.clongdouble)
                for j in range(n):
                    y += x[:, j] * A[i, j]
                term *= y
            tot += term.sum()
            size += np.abs(term).sum()
        rel = abs(est[b] - tot / iters) / (size / iters)
        _say(f"order {n}, couplings 2^-{k}: {float(rel):.2e}")
        assert rel <= (4 * n + 100) * 2.0 ** -53, (n, k, rel)


def test_gurvits_many_matrices_in_chunks(gpu):
    """More matrices than the fragments of one chunk: the ones around its end and
    one that keeps the FP64 products in the second chunk, against the oracle as
    in test_gurvits_batch_vs_oracle; and a call of few draws per matrix, which
    takes the FP64 products throughout, draws the same samples."""
    from perceval_amd.permanent import gurvits
    rng = np.random.RandomState(2)
    n, count, iters = 17, 5600, 700
    base = (rng.randn(40, n, n) + 1j * rng.randn(40, n, n)) / np.sqrt(n)
    mats = [base[b % 40] for b in range(count)]
    mats[5500] = mats[5500].copy()
    mats[5500][2, 3] = 2.0 ** -50
    check = [0, 1, 5459, 5460, 5461, 5462, 5500, count - 1]
    est, err = gurvits(mats, iters, seed=4, stream0=9)
    few, _ = gurvits([mats[b] for b in check[:2]], iters, seed=4, stream0=9)
    assert np.max(np.abs(few - est[:2]) / np.abs(est[:2])) < 1e-11
    for b in check:
        ref_est, ref_err = oracle.gurvits(mats[b], iters, seed=4, stream=9 + b)
        scale = max(ref_err * np.sqrt(iters) / 2.5758293035489004, abs(ref_est))
        assert abs(est[b] - ref_est) <= 1e-11 * scale, (b, est[b], ref_est)
        assert abs(err[b] - ref_err) <= 1e-6 * ref_err, (b, err[b], ref_err)
