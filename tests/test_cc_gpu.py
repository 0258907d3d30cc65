"""GPU parity of the Clifford & Clifford sampler.

The GPU and the oracle draw from the same counter-based uniforms, so for the
same seed they produce the same samples except where a uniform falls within
rounding distance of a CDF boundary; the statistical checks then compare with
exact distributions (small sizes) and closed-form moments (m=60, n=20)."""
import itertools
import math
from collections import Counter

import numpy as np
import pytest

import oracle
from perceval_amd.utils.workloads import haar_unitary

pytestmark = pytest.mark.gpu


def _say(msg):
    print(f"[cc-gpu] {msg}", flush=True)


@pytest.mark.parametrize("m,inp", [(8, [1, 1, 1, 1, 0, 0, 0, 0]), (6, [2, 0, 1, 0, 0, 1]), (3, [0, 0, 1])])
def test_same_seed_same_samples(gpu, m, inp):
    from perceval_amd.sampling import cc_samples
    U = haar_unitary(m, seed=m)
    g = cc_samples(U, inp, 2000, seed=99)
    c = oracle.cc_samples(U, inp, 2000, seed=99)
    assert (g.sum(axis=1) == sum(inp)).all()
    same = np.mean(np.all(g == c, axis=1))
    assert same >= 0.999, same


@pytest.mark.parametrize("m,n,count", [(1, 12, 4), (2, 16, 400), (3, 11, 2000), (4, 17, 400), (9, 10, 2000),
                                       (12, 15, 800), (12, 16, 400), (40, 17, 200), (6, 22, 60)])
def test_same_seed_same_samples_repeated_rows(gpu, m, n, count):
    """Photons that share modes are summed by multiplicity from step 10 on
    (slices from step 16): from all photons in one mode (no unique row, units
    of one term) to mostly distinct ones, the oracle's samples seed for seed."""
    from perceval_amd.sampling import cc_samples
    U = haar_unitary(m, seed=10 * m + n)
    inp = [n // m + (1 if i < n % m else 0) for i in range(m)]
    g = cc_samples(U, inp, count, seed=17)
    c = oracle.cc_samples(U, inp, count, seed=17)
    assert np.array_equal(g, c), np.nonzero(np.any(g != c, axis=1))[0][:10]


@pytest.mark.parametrize("m", [1, 5, 15, 16, 17, 32, 33, 64, 65])
def test_same_seed_same_samples_first_steps(gpu, m):
    """Steps 1..9 run in one launch up to 64 modes, 16 lanes a sample: photon
    numbers 1..10, modes around multiples of 16 and both sides of 32 and 64,
    repeated rows, and a count that is no multiple of the samples per block."""
    from perceval_amd.sampling import cc_samples, cc_samples_multi_device
    U = haar_unitary(m, seed=7 * m)
    inputs = [[n // m + (1 if i < n % m else 0) for i in range(m)] for n in range(1, 11)]
    multi = cc_samples_multi_device(U, inputs, [37] * 10, seed=21, first_sample=5).cpu().numpy()
    for n, inp in enumerate(inputs, 1):
        g = cc_samples(U, inp, 37, seed=21, first_sample=5 + 37 * (n - 1))
        c = oracle.cc_samples(U, inp, 37, seed=21, first_sample=5 + 37 * (n - 1))
        assert np.array_equal(g, c), (n, np.nonzero(np.any(g != c, axis=1))[0][:10])
        assert np.array_equal(multi[37 * (n - 1):37 * n], c), n


def test_same_seed_same_samples_m60_n20(gpu):
    from perceval_amd.sampling import cc_samples
    U = haar_unitary(60, seed=60)
    inp = [1] * 20 + [0] * 40
    _say("GPU 48 samples")
    g = cc_samples(U, inp, 48, seed=5, first_sample=1000)
    _say("oracle 48 samples")
    c = oracle.cc_samples(U, inp, 48, seed=5, first_sample=1000)
    _say("done")
    assert np.mean(np.all(g == c, axis=1)) >= 0.97


@pytest.mark.parametrize("n,count", [(26, 8), (28, 1)])
def test_same_seed_same_samples_up_to_28_photons(gpu, n, count):
    """Steps above 20 photons run split over many waves per sample (2^{k-20}
    parts of the 2^{k-2} Gray-code terms): the oracle's samples, seed for
    seed, at 26 and 28 photons (one sample at 28: a single sample fills the
    device)."""
    from perceval_amd.sampling import cc_samples
    m = n + 10
    U = haar_unitary(m, seed=m)
    inp = [1] * n + [0] * 10
    _say(f"GPU {count} samples, n={n}")
    g = cc_samples(U, inp, count, seed=7)
    _say(f"oracle {count} samples, n={n}")
    c = oracle.cc_samples(U, inp, count, seed=7)
    _say("done")
    assert (g.sum(axis=1) == n).all()
    assert np.array_equal(g, c)


@pytest.mark.parametrize("n,count", [(22, 6), (30, 2)])
def test_split_steps_do_not_depend_on_the_call(gpu, n, count):
    """A sample's draws depend on (seed, sample index) only: one call of
    `count` samples equals `count` calls of one sample each (first_sample
    set), with the split steps cut the same way in both, up to 30 photons."""
    from perceval_amd.sampling import cc_samples
    m = n + 8
    U = haar_unitary(m, seed=3 * m)
    inp = [1] * n + [0] * 8
    _say(f"n={n}: one call of {count}")
    together = cc_samples(U, inp, count, seed=11)
    _say(f"n={n}: {count} calls of one")
    apart = np.concatenate([cc_samples(U, inp, 1, seed=11, first_sample=i) for i in range(count)])
    assert (together.sum(axis=1) == n).all()
    assert np.array_equal(together, apart)


def test_many_short_slices_do_not_depend_on_the_call(gpu):
    """So many slices that waves take several at a time and keep a sample's rows
    between them: the samples of calls that take them one by one."""
    from perceval_amd.sampling import cc_samples
    m, n, count = 24, 16, 60000
    U = haar_unitary(m, seed=8)
    inp = [1] * n + [0] * (m - n)
    together = cc_samples(U, inp, count, seed=3)
    for first in (0, 31234, count - 500):
        assert np.array_equal(cc_samples(U, inp, 500, seed=3, first_sample=first), together[first:first + 500])


@pytest.mark.parametrize("inp", [[1, 1, 0, 1, 0], [2, 1, 0, 0]])
def test_distribution_chi_square(gpu, inp):
    from perceval_amd.sampling import cc_samples
    U = haar_unitary(len(inp), seed=13)
    exact = oracle.distribution_exact(U, inp)
    N = 50000
    s = cc_samples(U, inp, N, seed=17)
    cnt = Counter(map(tuple, s.tolist()))
    chi2, dof = 0.0, -1
    for st, p in exact.items():
        if p * N >= 5:
            chi2 += (cnt.get(st, 0) - p * N) ** 2 / (p * N)
            dof += 1
    z = ((chi2 / dof) ** (1 / 3) - (1 - 2 / (9 * dof))) / math.sqrt(2 / (9 * dof))
    assert z < 3.7, (chi2, dof)


def test_moments_m60_n20(gpu):
    from perceval_amd.sampling import cc_samples
    m = 60
    U = haar_unitary(m, seed=600)
    inp = [1] * 20 + [0] * 40
    N = 4000
    _say(f"GPU {N} samples m=60 n=20")
    s = cc_samples(U, inp, N, seed=11).astype(float)
    _say("done")
    assert (s.sum(axis=1) == 20).all()
    mean = (np.abs(U[:, :20]) ** 2).sum(axis=1)
    se = np.sqrt(np.maximum(s.var(axis=0), 1e-4) / N)
    assert np.all(np.abs(s.mean(axis=0) - mean) < 5 * se)
    # pair moments on a few mode pairs
    rng = np.random.RandomState(0)
    for j, k in rng.choice(m, size=(8, 2), replace=False):
        exp = sum(abs(U[j, i] * U[k, i2] + U[j, i2] * U[k, i]) ** 2 for i, i2 in itertools.combinations(range(20), 2))
        x = s[:, j] * s[:, k]
        assert abs(x.mean() - exp) < 5 * max(x.std(), 1e-3) / math.sqrt(N)


def test_deterministic_replay(gpu):
    from perceval_amd.sampling import cc_samples
    U = haar_unitary(10, seed=1)
    a = cc_samples(U, [1] * 5 + [0] * 5, 500, seed=3)
    b = cc_samples(U, [1] * 5 + [0] * 5, 500, seed=3)
    c = cc_samples(U, [1] * 5 + [0] * 5, 500, seed=4)
    assert np.array_equal(a, b)
    assert not np.array_equal(a, c)


def test_cc_samples_multi_equals_single_input_calls(gpu):
    """Rows of input i equal pcvl_cc_samples on input i with first_sample +
    row0_i, bit for bit (same counter streams), across photon numbers."""
    from perceval_amd.sampling import cc_samples, cc_samples_multi_device
    m = 10
    U = haar_unitary(m, seed=101)
    inputs = [[1, 1, 1, 1, 0, 0, 0, 0, 0, 0], [1, 1, 1, 0, 0, 0, 0, 0, 0, 0], [0] * m,
              [2, 0, 1, 0, 0, 0, 0, 0, 0, 1], [1, 0, 1, 1, 0, 0, 0, 0, 0, 0], [0, 0, 0, 0, 0, 0, 0, 0, 0, 5]]
    counts = [300, 257, 5, 0, 64, 100]
    seed, first = 4242, 1000
    out = cc_samples_multi_device(U, inputs, counts, seed=seed, first_sample=first).cpu().numpy()
    assert out.shape == (sum(counts), m)
    row = 0
    for inp, c in zip(inputs, counts):
        ref = cc_samples(U, inp, c, seed=seed, first_sample=first + row)
        assert np.array_equal(out[row:row + c], ref), inp
        assert (out[row:row + c].sum(axis=1) == sum(inp)).all()
        row += c
    # and seed for seed with the oracle on one of them
    row0 = counts[0] + counts[1] + counts[2] + counts[3]
    ref = oracle.cc_samples(U, inputs[4], counts[4], seed=seed, first_sample=first + row0)
    assert np.array_equal(out[row0:row0 + counts[4]], ref)


def test_backend_samples_for_inputs(gpu):
    from perceval_amd.backends import BackendFactory
    from perceval_amd.components import Unitary
    from perceval_amd.utils.states import BasicState
    U = haar_unitary(6, seed=7)
    b = BackendFactory.get_backend("CliffordClifford2017")
    b.set_circuit(Unitary(U))
    want = {BasicState([1, 1, 0, 0, 0, 0]): 50, BasicState([1, 0, 1, 0, 0, 0]): 20, BasicState([0, 0, 0, 0, 0, 0]): 3}
    got = b.samples_for_inputs(want)
    assert list(got) == list(want)
    for s, c in want.items():
        assert len(got[s]) == c
        assert all(o.n == s.n and o.m == 6 for o in got[s])
    with pytest.raises(AssertionError):
        b.samples_for_inputs({BasicState([1, 1, 0]): 2})


@pytest.mark.parametrize("m,n", [(20, 14), (24, 15), (66, 15)])
def test_one_wave_per_sample_and_slices_agree(gpu, m, n):
    """Steps 14 and 15 run in one wave per sample or in slices by the number of
    samples: the same samples, and the oracle's seed for seed."""
    from perceval_amd.sampling import cc_samples
    U = haar_unitary(m, seed=m + n)
    inp = [1] * n + [0] * (m - n)
    count = 8200
    sliced = cc_samples(U, inp, count, seed=6)
    assert np.array_equal(cc_samples(U, inp, 8192, seed=6), sliced[:8192])
    assert np.array_equal(cc_samples(U, inp, 8, seed=6, first_sample=8192), sliced[8192:])
    assert np.array_equal(oracle.cc_samples(U, inp, 40, seed=6), sliced[:40])


@pytest.mark.parametrize("m,n,counts", [(32, 15, (511, 512)), (33, 16, (511, 512, 4096, 4097)), (65, 15, (3, 4))])
def test_step_15_in_one_wave_or_in_slices(gpu, m, n, counts):
    """The sample counts between which step 15 changes its kernel, above 32 and
    above 64 modes: the same samples on both sides, in a workspace of the size
    that the library names."""
    from perceval_amd.sampling import cc_samples
    U = haar_unitary(m, seed=m + n)
    inp = [1] * n + [0] * (m - n)
    ref = cc_samples(U, inp, max(counts), seed=8)
    assert np.array_equal(oracle.cc_samples(U, inp, 3, seed=8), ref[:3])
    for count in counts:
        assert np.array_equal(cc_samples(U, inp, count, seed=8), ref[:count])


@pytest.mark.parametrize("m,n", [(64, 13), (65, 10), (65, 13), (80, 14), (128, 11)])
def test_same_seed_same_samples_row_by_row(gpu, m, n):
    """Above 64 modes, steps 10..13 sum every row by itself, repeated ones too."""
    from perceval_amd.sampling import cc_samples
    U = haar_unitary(m, seed=m * n)
    inp = [2, 1] + [1] * (n - 3) + [0] * (m - n + 1)
    assert np.array_equal(cc_samples(U, inp, 150, seed=2), oracle.cc_samples(U, inp, 150, seed=2))


@pytest.mark.parametrize("n,count", [(14, 8300), (17, 300), (21, 40)])
def test_smaller_workspaces_give_the_same_samples(gpu, n, count):
    """Any workspace from the least size on is taken, with fewer samples of the
    sliced steps at a time; one byte less than the least is refused."""
    import ctypes
    import torch
    from perceval_amd import _native
    from perceval_amd.sampling import cc_samples
    lib = _native.load()
    m = 24
    U = haar_unitary(m, seed=n)
    inp = np.array([1] * n + [0] * (m - n), dtype=np.int32)
    ref = cc_samples(U, inp, count, seed=4)
    full, least = ctypes.c_size_t(), ctypes.c_size_t()
    _native.check(lib.pcvl_cc_workspace_bytes(n, count, ctypes.byref(full)), "bytes")
    _native.check(lib.pcvl_cc_workspace_least_bytes(n, count, ctypes.byref(least)), "least")
    assert least.value < full.value
    dU = torch.from_numpy(U).cuda()
    work = torch.empty(full.value, dtype=torch.uint8, device="cuda")
    for size in (least.value, (least.value + full.value) // 2, full.value):
        out = torch.empty((count, m), dtype=torch.int32, device="cuda")
        rc = lib.pcvl_cc_samples(_native.ptr(dU), m, inp.ctypes.data_as(ctypes.POINTER(ctypes.c_int32)), count, 4, 0,
                                 _native.ptr(out), _native.ptr(work), size, _native.stream_handle())
        assert rc == 0 and np.array_equal(out.cpu().numpy(), ref), size
    assert lib.pcvl_cc_samples(_native.ptr(dU), m, inp.ctypes.data_as(ctypes.POINTER(ctypes.c_int32)), count, 4, 0,
                               _native.ptr(out), _native.ptr(work), least.value - 1, _native.stream_handle()) != 0


def test_sampling_on_a_nearly_full_device(gpu):
    """Where the whole workspace (44 MB here) does not fit, a smaller one is taken."""
    import torch
    from perceval_amd.sampling import cc_samples_device
    m, n, count = 24, 21, 2000
    dU = torch.from_numpy(haar_unitary(m, seed=n)).cuda()
    inp = [1] * n + [0] * (m - n)
    ref = cc_samples_device(dU, inp, count, seed=4).cpu().numpy()
    torch.cuda.empty_cache()
    room = torch.cuda.memory_reserved() + (24 << 20)
    try:
        torch.cuda.set_per_process_memory_fraction(room / torch.cuda.get_device_properties(0).total_memory)
        with pytest.raises(torch.OutOfMemoryError):
            torch.empty(40 << 20, dtype=torch.uint8, device="cuda")
        got = cc_samples_device(dU, inp, count, seed=4)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert np.array_equal(got.cpu().numpy(), ref)
