"""GPU parity of the HIP path against the CPU oracle, through the C-ABI.

Bars: class vectors, stop iterations and difference counts bit-exact; W, H and the KL
divergence within 1e-3 relative of the FP64 oracle (single half-steps: 1e-5)."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from conftest import GOLDEN, rel_err

pytestmark = pytest.mark.gpu

KS = [1, 2, 3, 4, 5, 7, 8, 10, 12, 16, 17, 20, 24, 28, 32, 33, 40, 48, 56, 64]


def make_job(nmfk, orc, n, m, k, seed_v=1, seed_init=2, mu=0.0, sigma=1.0):
    V = orc.gen_lognormal(n, m, seed_v, mu, sigma)
    job = nmfk.Job(n, m, k)
    job.set_V(V)
    job.init_random(seed_init)
    return job, V


def test_uniform_init_is_bit_exact(nmfk, orc):
    for n, m, k in [(100, 37, 3), (513, 64, 16), (70, 300, 33)]:
        with nmfk.Job(n, m, k) as job:
            job.init_random(77)
            W0, H0 = orc.init_WH(n, m, k, 77)
            assert np.array_equal(job.get_W(), W0)
            assert np.array_equal(job.get_H(), H0)


def test_V_roundtrip_and_generators(nmfk, orc):
    n, m = 257, 131
    V = orc.gen_lognormal(n, m, 3, 5.0, 1.5)
    with nmfk.Job(n, m, 4) as job:
        job.set_V(V)
        assert np.array_equal(job.get_V(), V)
        job.gen_V_lognormal(3, 5.0, 1.5)
        assert rel_err(job.get_V(), V) < 1e-6          # device libm vs host libm, FP64 then rounded
        job.gen_V_planted(4, 6, 0.3)
        assert rel_err(job.get_V(), orc.gen_planted(n, m, 6, 4, 0.3)) < 1e-6


# Tolerance of one half-step against the FP64 oracle: FP32 arithmetic 1e-5; BF16
# contractions (8-bit significands, FP32 accumulation) 1e-2.
def half_tol(job):
    return 1e-2 if job.kernel_path() == 3 else 1e-5


@pytest.mark.parametrize("path", [0, 1, 2, 3])
@pytest.mark.parametrize("k", KS)
def test_half_steps_match_oracle(nmfk, orc, k, path):
    # path 0: automatic (at 700 x 150 FP32 matrix cores up to k = 32, ranks up to 8 padded to
    # 16; BF16 matrix cores above), 1: vector ALUs, 2: FP32 matrix cores, 3: BF16 matrix cores
    # (each falls back to the next simpler path where the padded rank does not fit it).
    n, m = 700, 150
    job, V = make_job(nmfk, orc, n, m, k, seed_v=k, seed_init=k + 100)
    with job:
        job.set_kernel_path(path)
        tol = half_tol(job)
        W0, H0 = orc.init_WH(n, m, k, k + 100)
        job.update_H()
        H1 = orc.update_H(V, W0, H0)
        assert rel_err(job.get_H(), H1) < tol
        job.update_W()
        W1 = orc.update_W(V, W0, H1)
        assert rel_err(job.get_W(), W1) < tol


@pytest.mark.parametrize("n,m,k", [(1, 1, 1), (5, 3, 2), (63, 65, 3), (1000, 7, 7), (9, 2000, 2),
                                   (17, 33, 9), (100, 13, 13), (31, 1100, 20), (2000, 47, 40)])
def test_half_steps_ragged_shapes(nmfk, orc, n, m, k):
    job, V = make_job(nmfk, orc, n, m, k, seed_v=n + m, seed_init=k)
    with job:
        W0, H0 = orc.init_WH(n, m, k, k)
        for _ in range(3):
            job.update_H()
            H0 = orc.update_H(V, W0, H0)
            job.update_W()
            W0 = orc.update_W(V, W0, H0)
        tol = 2e-2 if job.kernel_path() == 3 else 1e-4
        assert rel_err(job.get_H(), H0) < tol
        assert rel_err(job.get_W(), W0) < tol


@pytest.mark.parametrize("na,nb", [(4, 1), (2, 2), (2, 4), (1, 4)])
@pytest.mark.parametrize("k", [3, 7])
def test_small_rank_shapes_match_oracle(nmfk, orc, k, na, nb):
    # Ranks up to 8 on the FP32 matrix cores: the rank is padded to 16, and both products sum
    # only the rank's own columns (GEMM2 in 4x4 blocks whose lane groups are added once per
    # split).  Every workgroup shape gives the FP64 oracle's half-steps: one wave group (no LDS
    # step, idle waves in the last workgroup at 700 rows) and two or four (LDS step), with
    # masked last blocks (1300 and 700 rows are not multiples of 16).
    n, m = 1300, 700
    old = (nmfk.tune_get(nmfk.TUNE_MFMA_NA), nmfk.tune_get(nmfk.TUNE_MFMA_NB))
    nmfk.tune_set(nmfk.TUNE_MFMA_NA, na)
    nmfk.tune_set(nmfk.TUNE_MFMA_NB, nb)
    try:
        job, V = make_job(nmfk, orc, n, m, k, seed_v=k + 7, seed_init=k + 8)
        with job:
            job.set_kernel_path(2)
            pl = job.plan()
            assert pl["H"]["nab"] == -(-m // (64 * na)) and pl["W"]["nab"] == -(-n // (64 * na)), pl
            for _ in range(2):   # each half-step from the device's own previous factors
                W, H = job.get_W(), job.get_H()
                job.update_H()
                assert rel_err(job.get_H(), orc.update_H(V, W, H)) < 1e-5
                H = job.get_H()
                job.update_W()
                assert rel_err(job.get_W(), orc.update_W(V, W, H)) < 1e-5
    finally:
        nmfk.tune_set(nmfk.TUNE_MFMA_NA, old[0])
        nmfk.tune_set(nmfk.TUNE_MFMA_NB, old[1])


@pytest.mark.parametrize("n,m,k", [(98311, 64, 17), (98400, 65, 32), (6465, 1000, 33), (1041, 6151, 64),
                                   (191000, 33, 24), (25601, 257, 48), (6465, 1000, 9), (6401, 1087, 16),
                                   (1087, 6401, 12)])
def test_split_products_match_oracle(nmfk, orc, n, m, k):
    # Jobs that run on products of three-part BF16 operands (nmfk_split_rule), at sizes around
    # the 16-row blocks, the 64-row tiles and the wave groups' shares: each half-step within the
    # FP32 bar of the oracle, and the FP32 instructions (the same job replanned to a workgroup
    # target) within the same bar.
    job, V = make_job(nmfk, orc, n, m, k, seed_v=n + m, seed_init=k)
    with job:
        job.set_kernel_path(2)
        W, H = orc.init_WH(n, m, k, k)
        H1 = orc.update_H(V, W, H)
        W1 = orc.update_W(V, W, H1)
        for target in (0, 1024):
            job.replan(target)
            job.set_WH(W, H)
            job.update_H()
            assert rel_err(job.get_H(), H1) < 1e-5
            job.update_W()
            assert rel_err(job.get_W(), W1) < 1e-5


@pytest.mark.parametrize("n,m,k", [(90001, 70, 12), (90001, 70, 24), (90001, 70, 48)])
def test_split_products_keep_infinities(nmfk, orc, n, m, k):
    # An infinite value of V makes its column's H row infinite, as on the FP32 instructions; the
    # other rows of H stay finite and right.
    V = orc.gen_lognormal(n, m, 3, 0.0, 1.0)
    W, H = orc.init_WH(n, m, k, 5)
    want = orc.update_H(V, W, H)
    V[100, 37] = np.inf
    with nmfk.Job(n, m, k) as job:
        job.set_V(V)
        job.init_random(5)
        job.set_kernel_path(2)
        job.update_H()
        got = job.get_H()
    assert np.all(np.isposinf(got[37]))
    keep = np.arange(m) != 37
    assert rel_err(got[keep], want[keep]) < 1e-5


@pytest.mark.parametrize("n,m,k", [(6401, 1087, 13), (98400, 65, 30)])
def test_split_products_same_bits_in_a_batch(nmfk, n, m, k):
    with nmfk.Job(n, m, k) as a, nmfk.Job(n, m, k) as b:
        batch = nmfk.Batch(5, 4)
        for j in (a, b):
            j.gen_V_lognormal(9, 0.0, 1.0)
            j.init_random(4)
        a.run(20, 5, 1000)
        batch.add(b, 20, 1000)
        batch.run()
        batch.close()
        assert np.array_equal(a.get_W(), b.get_W()) and np.array_equal(a.get_H(), b.get_H())


@pytest.mark.parametrize("n,m,k,path,na,nb", [
    (1985, 33, 3, 2, 1, 4), (2049, 64, 7, 2, 2, 2), (2111, 65, 16, 2, 4, 1), (1985, 40, 12, 2, 2, 4), (2305, 39, 30, 2, 4, 2),
    (2049, 65, 40, 2, 4, 2), (1985, 33, 20, 3, 2, 4), (2111, 63, 48, 3, 1, 4), (30, 5, 4, 1, 1, 4), (2047, 5, 5, 1, 1, 4),
    (65, 9, 7, 1, 1, 4), (2049, 20, 13, 1, 1, 4), (2001, 30, 20, 1, 1, 4), (32801, 40, 34, 1, 1, 4)])
def test_one_split_finishes_in_its_launch(nmfk, orc, n, m, k, path, na, nb):
    # A half-step of one split updates its rows, their column sums and BF16 copies in the launch
    # that sums them: two iterations, so that the second divides by those column sums, in every
    # workgroup shape and with partly filled last blocks of rows, against the FP64 oracle.  The
    # bar is four half-steps at the 1e-5 of one (BF16: that of the ragged shapes).
    old = (nmfk.tune_get(nmfk.TUNE_MFMA_NA), nmfk.tune_get(nmfk.TUNE_MFMA_NB))
    nmfk.tune_set(nmfk.TUNE_MFMA_NA, na)
    nmfk.tune_set(nmfk.TUNE_MFMA_NB, nb)
    try:
        job, V = make_job(nmfk, orc, n, m, k, seed_v=n + k, seed_init=k)
        with job:
            job.set_kernel_path(path)
            assert job.plan()["W"]["S"] == 1
            W, H = orc.init_WH(n, m, k, k)
            for _ in range(2):
                H = orc.update_H(V, W, H)
                W = orc.update_W(V, W, H)
            job.run(2, 2, 1000)
            tol = 2e-2 if path == 3 else 4e-5
            assert rel_err(job.get_H(), H) < tol and rel_err(job.get_W(), W) < tol
    finally:
        nmfk.tune_set(nmfk.TUNE_MFMA_NA, old[0])
        nmfk.tune_set(nmfk.TUNE_MFMA_NB, old[1])


@pytest.mark.parametrize("n,m,k,path", [(64, 33, 3, 2), (65, 1025, 7, 2), (1024, 63, 12, 2), (1025, 1024, 30, 2), (1023, 40, 5, 1),
                                        (30, 5, 4, 1), (1000, 70, 40, 3), (1024, 1023, 64, 2)])
def test_lone_half_steps_give_the_bits_of_a_run(nmfk, orc, n, m, k, path):
    # Half-steps called one by one take their denominators from the factor itself up to 1024 rows,
    # from its column-sum partials above: in both cases the sums a run's finishes leave behind.
    jobs = [make_job(nmfk, orc, n, m, k, seed_v=n, seed_init=m)[0] for _ in range(2)]
    with jobs[0] as a, jobs[1] as b:
        for j in jobs:
            j.set_kernel_path(path)
        a.run(2, 1000, 1000)
        for _ in range(2):
            b.update_H()
            b.update_W()
        assert np.array_equal(a.get_H(), b.get_H()) and np.array_equal(a.get_W(), b.get_W())


@pytest.mark.parametrize("n,m", [(16000, 256), (16000, 257)])
def test_lone_half_steps_of_one_split_give_the_bits_of_a_run(nmfk, orc, n, m):
    # W half-steps of one split on both sides of the line between denominators from H itself and from
    # its column sums.
    jobs = [make_job(nmfk, orc, n, m, 48, seed_v=n, seed_init=m)[0] for _ in range(2)]
    with jobs[0] as a, jobs[1] as b:
        assert a.kernel_path() == 3 and a.plan()["W"]["S"] == 1
        a.run(2, 1000, 1000)
        for _ in range(2):
            b.update_H()
            b.update_W()
        assert np.array_equal(a.get_H(), b.get_H()) and np.array_equal(a.get_W(), b.get_W())


def test_split_products_are_a_property_of_the_job(nmfk):
    # Automatic: by size and rank, for a job planned on its own.  On or off holds for every plan;
    # neither has an effect off the FP32 matrix cores, or at padded ranks below 32.
    with nmfk.Job(6401, 1087, 20) as big, nmfk.Job(700, 150, 48) as small, nmfk.Job(6401, 1087, 16) as low:
        assert big.split() and not small.split() and not low.split()
        low.set_split(low.SPLIT_ON)
        assert not low.split()
        big.replan(1024)
        assert not big.split()
        big.set_split(big.SPLIT_ON)
        assert big.split()
        big.set_split(big.SPLIT_OFF)
        for target in (0, 8, 1024):
            big.replan(target)
            assert not big.split()
        big.set_split(big.SPLIT_AUTO)
        big.replan(0)
        assert big.split()
        big.set_kernel_path(1)
        assert not big.split()
        big.set_split(big.SPLIT_ON)
        assert not big.split()
        big.set_kernel_path(2)
        assert big.split()
        small.set_split(small.SPLIT_ON)
        assert small.kernel_path() == 3 and not small.split()
        small.set_kernel_path(2)
        assert small.split()
        for mode in (-1, 3):
            with pytest.raises(nmfk.NmfkError):
                big.set_split(mode)
    V = np.ones((64, 40), np.float32)
    with nmfk.Job.streamed(V, 3) as job:
        assert not job.split()
        with pytest.raises(nmfk.NmfkError):
            job.set_split(job.SPLIT_ON)


@pytest.mark.parametrize("n,m,k,path", [(64, 33, 17, 2), (65, 1025, 20, 2), (1024, 63, 24, 2), (1025, 1024, 30, 2), (1000, 70, 20, 0),
                                        (1024, 1023, 64, 2), (1025, 70, 40, 2), (6401, 1087, 18, 0)])
def test_lone_split_half_steps_give_the_bits_of_a_run(nmfk, orc, n, m, k, path):
    # On split products the denominators always come from column-sum partials, added as trees by a
    # kernel of their own here and by the finishes in a run: the same sums.
    jobs = [make_job(nmfk, orc, n, m, k, seed_v=n, seed_init=m)[0] for _ in range(2)]
    with jobs[0] as a, jobs[1] as b:
        for j in jobs:
            j.set_kernel_path(path)
            j.set_split(j.SPLIT_ON)
            assert j.split()
        a.run(2, 1000, 1000)
        for _ in range(2):
            b.update_H()
            b.update_W()
        assert np.array_equal(a.get_H(), b.get_H()) and np.array_equal(a.get_W(), b.get_W())


@pytest.mark.parametrize("n,m,k", [(500000, 32, 24), (400000, 40, 40)])
def test_split_products_do_not_lose_long_sums(nmfk, orc, n, m, k):
    # Sums of thousands of rows per wave keep no bias: the mean relative error of an H half-step
    # stays below 2^-25.  Rounding to nearest leaves m k entries within 2^-23 and k denominators within
    # 2^-24 of their values, whose means are below 2^-25 by far; sums that lose a part of every
    # term reach 8e-8 here.
    with nmfk.Job(n, m, k) as job:
        job.set_kernel_path(2)
        assert job.split()
        job.gen_V_planted(3, 6, 0.3)
        job.init_random(4)
        W, H = job.get_W(), job.get_H()
        want = orc.update_H(job.get_V(), W, H).astype(np.float64)
        job.update_H()
        assert abs(np.mean(job.get_H() / want) - 1.0) < 2.0 ** -25


def each_rel_err(got, want):
    """Largest relative error of any single value."""
    return float(np.max(np.abs(got.astype(np.float64) - want) / np.maximum(np.abs(want), 1e-300)))


def split_half_steps(nmfk, orc, V, W, H):
    """Both half-steps on split products and in 64 bits, W from the device's own H."""
    n, m, k = *V.shape, W.shape[1]
    with nmfk.Job(n, m, k) as job:
        job.set_V(V)
        job.set_kernel_path(2)
        job.set_split(job.SPLIT_ON)
        assert job.split()
        job.set_WH(W, H)
        job.update_H()
        H1 = job.get_H()
        job.update_W()
        return H1, orc.update_H(V, W, H), job.get_W(), orc.update_W(V, W, H1)


@pytest.mark.parametrize("scale", [3e-37, 1e-35, 1e-33, 1e18, 1e24, 1e30])
@pytest.mark.parametrize("n,m,k", [(700, 150, 24), (333, 150, 20), (700, 65, 40)])
def test_split_products_at_any_scale_of_V(nmfk, orc, n, m, k, scale):
    # Every value of H and W, not only the large ones, within the FP32 bar of a half-step: ratios near
    # the lowest and products near the highest numbers.
    V = (orc.gen_lognormal(n, m, 3, 0.0, 0.5).astype(np.float64) * scale).astype(np.float32)
    W, H = orc.init_WH(n, m, k, 5)
    H1, want_H, W1, want_W = split_half_steps(nmfk, orc, V, W + np.float32(0.1), H + np.float32(0.1))
    assert each_rel_err(H1, want_H) < 1e-5 and each_rel_err(W1, want_W) < 1e-5


@pytest.mark.parametrize("n,m,k", [(700, 150, 24), (333, 150, 20), (700, 65, 40)])
def test_split_products_keep_tiny_factors(nmfk, orc, n, m, k):
    # Factors with components on their way to zero and at the clamp (1.18e-38): their columns of the
    # other factor come from sums of such values alone.
    rng = np.random.default_rng(n)
    V = orc.gen_lognormal(n, m, 3, 3.0, 0.5)
    W, H = (x + np.float32(0.1) for x in orc.init_WH(n, m, k, 5))
    W[:, 1] *= np.float32(1e-35)
    W[:, 3] = np.float32(1.17549435e-38)
    W[:, 4] = np.exp(rng.uniform(np.log(1e-36), np.log(1e-33), n)).astype(np.float32)
    H[rng.random(H.shape) < 0.2] = np.float32(1.17549435e-38)
    H[:, 5] *= np.float32(1e-34)
    H1, want_H, W1, want_W = split_half_steps(nmfk, orc, V, W, H)
    ok = np.abs(want_H) > 1e-36   # below, FP32 itself runs out of digits
    assert each_rel_err(H1[ok], want_H[ok]) < 1e-5
    ok = np.abs(want_W) > 1e-36
    assert each_rel_err(W1[ok], want_W[ok]) < 1e-5


@pytest.mark.parametrize("n,m,k", [(700, 150, 24), (333, 150, 20), (700, 65, 40)])
def test_split_products_of_large_factors(nmfk, orc, n, m, k):
    # Products of the factors of 1e29 and more against a V of about 1: ratios of 1e-30 that do not vanish.
    V = orc.gen_lognormal(n, m, 3, 0.0, 0.5)
    W, H = orc.init_WH(n, m, k, 5)
    W, H = (W + np.float32(0.1)) * np.float32(1e15), (H + np.float32(0.1)) * np.float32(3e14)
    H1, want_H, W1, want_W = split_half_steps(nmfk, orc, V, W, H)
    assert each_rel_err(H1, want_H) < 1e-5 and each_rel_err(W1, want_W) < 1e-5


@pytest.mark.parametrize("n,m,k", [(700, 150, 24), (333, 150, 20), (700, 65, 40)])
def test_split_products_with_an_empty_row_or_column(nmfk, orc, n, m, k):
    # A row of V without any value: its row of W goes to the clamp, and all others stay right (four
    # iterations at the bar of one half-step each).  A column without any makes its row of H zero, and
    # 0 / 0 in the W half-step: NaN where the FP32 instructions have it.
    V = orc.gen_lognormal(n, m, 3, 5.0, 1.0)
    V[17] = 0.0
    W, H = orc.init_WH(n, m, k, 5)
    ref = orc.nmf(V, W, H, 4, 1, 1000, fp64=True)
    with nmfk.Job(n, m, k) as job:
        job.set_V(V)
        job.set_kernel_path(2)
        job.set_split(job.SPLIT_ON)
        job.set_WH(W, H)
        job.run(4, 1, 1000)
        W1, H1 = job.get_W(), job.get_H()
        assert np.all(W1[17] == np.float32(1.17549435e-38))
        assert rel_err(H1, ref["H"]) < 4e-5 and rel_err(W1, ref["W"]) < 4e-5
        V[:, 9] = 0.0
        job.set_V(V)
        got = []
        for mode in (job.SPLIT_ON, job.SPLIT_OFF):
            job.set_split(mode)
            job.set_WH(W, H)
            job.update_H()
            assert np.all(job.get_H()[9] == 0.0)
            job.update_W()
            got.append(np.isnan(job.get_W()))
        assert got[0].any() and np.array_equal(*got)


@pytest.mark.parametrize("n,m,k,wide", [(900, 130, 30, 1), (12000, 1100, 30, 2)])
def test_split_products_same_bits_in_every_batch_class(nmfk, orc, n, m, k, wide):
    # 1 x 4 and (W halves of 1000-4095 columns and enough rows) 2 x 2 waves; split products at any size when asked for, beside a job on the FP32 instructions in the same batch.
    V = orc.gen_lognormal(n, m, 4, 0.0, 1.0)
    jobs = [nmfk.Job(n, m, k) for _ in range(4)]
    try:
        for i, j in enumerate(jobs):
            j.set_V(V)
            j.init_random(6)
            j.set_split(j.SPLIT_ON if i < 2 else j.SPLIT_OFF)
            assert j.split() == (i < 2) and j.plan()["W"]["nab"] == -(-n // (64 * wide))
        batch = nmfk.Batch(5, 4)
        batch.add(jobs[1], 10, 1000)
        batch.add(jobs[3], 10, 1000)
        batch.run()
        batch.close()
        for a, b in ((jobs[0], jobs[1]), (jobs[2], jobs[3])):
            a.run(10, 5, 1000)
            assert np.array_equal(a.get_W(), b.get_W()) and np.array_equal(a.get_H(), b.get_H())
        assert not np.array_equal(jobs[0].get_W(), jobs[2].get_W())
    finally:
        for j in jobs:
            j.close()


@pytest.mark.parametrize("n,m,k", [(6401, 1087, 13), (98400, 65, 9), (25601, 257, 16), (12000, 1100, 12)])
def test_tree_sums_at_padded_rank_16_give_the_same_bits(nmfk, n, m, k):
    # Alone, by half-steps and in a batch, beside a job that adds in ascending order.
    jobs = [nmfk.Job(n, m, k) for _ in range(5)]
    try:
        for i, j in enumerate(jobs):
            j.gen_V_lognormal(n, 0.0, 1.0)
            j.init_random(m)
            j.set_split(j.SPLIT_OFF if i >= 3 else j.SPLIT_AUTO)
            assert not j.split()
        a, b, c, d, e = jobs
        batch = nmfk.Batch(5, 4)
        batch.add(b, 10, 1000)
        batch.add(e, 10, 1000)
        batch.run()
        batch.close()
        for x, y in ((a, b), (d, e)):
            x.run(10, 5, 1000)
            assert np.array_equal(x.get_W(), y.get_W()) and np.array_equal(x.get_H(), y.get_H())
        assert not np.array_equal(a.get_W(), d.get_W())
        a.init_random(m)
        a.run(2, 1000, 1000)
        for _ in range(2):
            c.update_H()
            c.update_W()
        assert np.array_equal(a.get_W(), c.get_W()) and np.array_equal(a.get_H(), c.get_H())
        a.set_split(a.SPLIT_OFF)   # the captured interval of the trees is not run again
        for j in (a, d):
            j.init_random(m)
            j.run(10, 5, 1000)
        assert np.array_equal(a.get_W(), d.get_W()) and np.array_equal(a.get_H(), d.get_H())
    finally:
        for j in jobs:
            j.close()


@pytest.mark.parametrize("n,m,k", [(98400, 65, 9), (200000, 40, 14)])
def test_tree_sums_at_padded_rank_16_are_nearer_to_64_bits(nmfk, n, m, k):
    # Four ascending chains of n / 256 column-sum partials each err by about sqrt(n / 768) / 2
    # roundings, trees of 8 by a third of that.
    errs = []
    for mode in (0, 1):
        with nmfk.Job(n, m, k) as job:
            job.set_split(mode)
            job.gen_V_planted(3, 6, 0.3)
            job.init_random(4)
            V, W, H = (x.astype(np.float64) for x in (job.get_V(), job.get_W(), job.get_H()))
            job.update_H()
            want = H * ((V / (W @ H.T)).T @ W) / W.sum(axis=0)
            errs.append(np.sqrt(np.mean((job.get_H() / want - 1.0) ** 2)))
    assert errs[0] < errs[1], errs


def test_golden_tiny_runs(nmfk, orc):
    g = np.load(GOLDEN / "tiny.npz")
    for ci in range(int(g["ncases"])):
        p = f"c{ci}_"
        n, m, k, sv, si = (int(x) for x in g[p + "shape"])
        with nmfk.Job(n, m, k) as job:
            job.set_V(g[p + "V"])
            job.init_random(si)
            job.set_kernel_path(2 if k > 8 else 0)   # FP32 arithmetic: the reference's precision
            r = job.run(200, 5, 3)
            assert r["iterations"] == int(g[p + "iterations"]), ci
            assert r["converged"] == bool(g[p + "converged"]) and r["ntests"] == int(g[p + "ntests"])
            assert np.array_equal(job.get_classification(), g[p + "cls"]), ci


def test_config0_parity(nmfk, orc):
    # V 5000x38 lognormal(5, 1.5^2), k=3, T=10, stop_threshold=40, 2000 iterations.
    g = np.load(GOLDEN / "config0.npz")
    n, m, k, sv, si = (int(x) for x in g["params"])
    V = orc.gen_lognormal(n, m, sv, 5.0, 1.5)
    with nmfk.Job(n, m, k) as job:
        job.set_V(V)
        job.init_random(si)
        r = job.run(2000, 10, 40)
        assert r["converged"] and r["iterations"] == int(g["f64_iterations"])
        assert np.array_equal(job.get_classification(), g["f64_cls"])
        assert rel_err(job.get_H(), g["f64_H"]) < 1e-3
        assert rel_err(job.get_W()[:64], g["f64_W_head"]) < 1e-3
        _, _, kl = job.dot_kl()
        assert abs(kl - float(g["f64_kl"])) / float(g["f64_kl"]) < 1e-3


def test_run_equals_reference_structured_steps(nmfk, orc):
    # nmfk_job_run (graph-captured intervals, column sums fused into the finish kernel,
    # clamps in-register) must give the same bits as update_H/update_W/adjust.
    n, m, k, T = 900, 120, 6, 4
    V = orc.gen_lognormal(n, m, 5, 0.0, 1.0)
    with nmfk.Job(n, m, k) as a, nmfk.Job(n, m, k) as b:
        for j in (a, b):
            j.set_V(V)
            j.init_random(9)
        a.run(3 * T + 2, T, 1000)
        for _ in range(3):
            for _ in range(T):
                b.update_H()
                b.update_W()
            b.adjust()
        for _ in range(2):
            b.update_H()
            b.update_W()
        assert np.array_equal(a.get_W(), b.get_W())
        assert np.array_equal(a.get_H(), b.get_H())


def test_matrix_core_and_vector_paths_agree(nmfk, orc):
    n, m, k = 2500, 300, 16
    V = orc.gen_lognormal(n, m, 8, 0.0, 1.0)
    res = []
    for path in (1, 2):
        with nmfk.Job(n, m, k) as j:
            j.set_V(V)
            j.init_random(4)
            j.set_kernel_path(path)
            assert j.kernel_path() == path
            r = j.run(200, 10, 5)
            res.append((r, j.get_classification(), j.get_W(), j.get_H()))
    (r1, c1, W1, H1), (r2, c2, W2, H2) = res
    assert r1["iterations"] == r2["iterations"] and np.array_equal(c1, c2)
    assert rel_err(W2, W1) < 1e-3 and rel_err(H2, H1) < 1e-3


def test_runs_are_deterministic(nmfk, orc):
    n, m, k = 3000, 400, 16
    V = orc.gen_lognormal(n, m, 6, 0.0, 1.0)
    outs = []
    for _ in range(2):
        with nmfk.Job(n, m, k) as j:
            j.set_V(V)
            j.init_random(1)
            j.run(40, 10, 1000)
            outs.append((j.get_W(), j.get_H()))
    assert np.array_equal(outs[0][0], outs[1][0]) and np.array_equal(outs[0][1], outs[1][1])


def test_dot_and_kl_match_oracle(nmfk, orc):
    n, m, k = 500, 90, 5
    job, V = make_job(nmfk, orc, n, m, k)
    with job:
        job.run(30, 10, 100)
        W, H = job.get_W(), job.get_H()
        dv, dvwh, kl = job.dot_kl()
        odv, odvwh = orc.dot_VWH(V.astype(np.float64), W.astype(np.float64), H.astype(np.float64))
        okl = orc.kl_div(V, W, H, fp64=True)
        assert abs(dv - odv) / odv < 1e-12
        assert abs(dvwh - odvwh) / odvwh < 1e-9
        assert abs(kl - okl) / okl < 1e-9


@pytest.mark.parametrize("n,m,k", [(1, 1, 1), (16, 64, 4), (17, 65, 9), (333, 20, 8), (1023, 257, 16), (50, 5003, 20),
                                   (2049, 70, 33)])
def test_dot_kl_matches_float64(nmfk, orc, n, m, k):
    # Sizes around the 16-row blocks, the 64-column waves and the 256-column workgroups, V with
    # zeros, values of 60 orders of magnitude; a zero product under a positive value gives an
    # infinite divergence.
    rng = np.random.default_rng(n + m)
    V = np.exp(rng.normal(0.0, 20.0, (n, m))).clip(0, 1e18).astype(np.float32)
    V[rng.random((n, m)) < 0.1] = 0.0
    W, H = orc.init_WH(n, m, k, 3)
    with nmfk.Job(n, m, k) as job:
        W0 = W.copy()
        W0[0] = 0.0
        V[0, 0] = 1.0
        job.set_V(V)
        job.set_WH(W0, H)
        assert job.dot_kl()[2] == np.inf
    V[0, 0] = 0.0
    v, wh = V.astype(np.float64), W.astype(np.float64) @ H.T.astype(np.float64)
    with nmfk.Job(n, m, k) as job:
        job.set_V(V)
        job.set_WH(W, H)
        got = job.dot_kl()
    kl = np.where(v > 0, v * np.log(np.where(v > 0, v, 1.0) / wh), 0.0) - v + wh
    want = (np.sum(v * v), np.sum((v - wh) ** 2), np.sum(kl))
    scale = (want[0], want[1], np.sum(np.abs(kl)))
    for a, b, c in zip(got, want, scale):
        assert abs(a - b) <= 1e-12 * c + 1e-300


def test_stop_rule_on_device_matches_oracle_trace(nmfk, orc):
    # Per-test differences counted on the device (contingency table) reproduce the
    # oracle's pairwise count through the whole run, including the reset cases.
    # Compared test by test: src/common.c:1195-1209 is integer work, so every count must be
    # equal, the non-zero ones included (a count that only kept the zero pattern would fail).
    n, m, k = 400, 60, 4
    V = orc.gen_lognormal(n, m, 12, 0.0, 1.0)
    W0, H0 = orc.init_WH(n, m, k, 13)
    o = orc.nmf(V, W0, H0, 600, 3, 6, fp64=True, max_trace=400)
    with nmfk.Job(n, m, k) as job:
        job.set_V(V)
        job.init_random(13)
        r = job.run(600, 3, 6, trace=True)
        assert r["iterations"] == o["iterations"] and r["ntests"] == o["ntests"]
        assert np.array_equal(job.get_classification(), o["cls"])
        dev, ref = r["diff_trace"], o["diff_trace"]
        assert len(dev) == r["ntests"] == len(ref)
        assert np.array_equal(dev, ref), np.nonzero(dev != ref)
        assert r["last_diff"] == ref[-1]
        nz = np.count_nonzero(ref)
        assert nz >= 3 and len(set(ref[ref > 0].tolist())) >= 2   # several distinct non-zero counts


@pytest.mark.parametrize("n,m,k,seed", [(3000, 97, 3, 41), (1200, 300, 7, 42), (2500, 150, 12, 43),
                                        (3000, 30, 5, 44)])
def test_device_difference_counts_equal_oracle(nmfk, orc, n, m, k, seed):
    # Larger m (more pairs, up to 44850) and both kernel families (matrix cores at padded rank
    # 16, the vector ALUs at kt 8 on the 30-column V): the device's per-test differences equal
    # the FP64 oracle's pairwise counts.
    V = orc.gen_lognormal(n, m, seed, 5.0, 1.5)
    W0, H0 = orc.init_WH(n, m, k, seed + 100)
    o = orc.nmf(V, W0, H0, 400, 10, 40, fp64=True, max_trace=100)
    with nmfk.Job(n, m, k) as job:
        job.set_V(V)
        job.init_random(seed + 100)
        r = job.run(400, 10, 40, trace=True)
    assert r["ntests"] == o["ntests"] == 40
    assert np.array_equal(r["diff_trace"], o["diff_trace"]), (r["diff_trace"], o["diff_trace"])
    assert np.count_nonzero(o["diff_trace"]) >= 2


def test_full_size_config1_shape(nmfk, orc):
    # 20000 x 1000, k = 16, planted rank 16: two iterations against the FP64 oracle, then
    # size-independent properties over 30 more (KL non-increasing, factors finite >= 0).
    n, m, k = 20000, 1000, 16
    V = orc.gen_planted(n, m, 16, 21, 0.3)
    W0, H0 = orc.init_WH(n, m, k, 22)
    with nmfk.Job(n, m, k) as job:
        job.set_V(V)
        job.init_random(22)
        W, H = W0.astype(np.float64), H0.astype(np.float64)
        for _ in range(2):
            job.update_H()
            job.update_W()
            H = orc.update_H(V, W, H)
            W = orc.update_W(V, W, H)
        assert rel_err(job.get_H(), H) < 1e-4 and rel_err(job.get_W(), W) < 1e-4
        prev = job.dot_kl()[2]
        for _ in range(3):
            job.run(10, 10, 1000)
            cur = job.dot_kl()[2]
            assert cur <= prev * (1 + 1e-6)
            prev = cur
        for A in (job.get_W(), job.get_H()):
            assert np.all(np.isfinite(A)) and A.min() >= 0


def test_bf16_path_error_against_fp64(nmfk, orc):
    # BF16 contractions with FP32 accumulation at k = 40 (padded to 64): 60 iterations from
    # the same start as the FP64 oracle.  Stated errors: relative Frobenius error of W.H,
    # relative KL difference, and class-vector agreement.
    n, m, k, iters = 3000, 400, 40, 60
    V = orc.gen_planted(n, m, 48, 77, 0.3)
    W0, H0 = orc.init_WH(n, m, k, 5)
    o = orc.nmf(V, W0, H0, iters, 10, 1000, fp64=True)
    with nmfk.Job(n, m, k) as j:
        j.set_V(V)
        j.init_random(5)
        assert j.kernel_path() == 3
        r = j.run(iters, 10, 1000)
        assert r["iterations"] == iters
        W, H = j.get_W().astype(np.float64), j.get_H().astype(np.float64)
        cls = j.get_classification()
    WH, WHo = W @ H.T, o["W"] @ o["H"].T
    fro = float(np.linalg.norm(WH - WHo) / np.linalg.norm(WHo))
    kl, klo = orc.kl_div(V, W, H), orc.kl_div(V, o["W"], o["H"])
    agree = float(np.mean(cls == orc.idx_max(o["H"])))
    print(f"bf16 k={k}: rel Frobenius(WH) {fro:.3e}, rel KL diff {abs(kl - klo) / klo:.3e}, class agreement {agree:.3f}")
    assert fro < 2e-2
    assert abs(kl - klo) / klo < 1e-2
    assert agree > 0.8


@pytest.mark.parametrize("k", [16, 24])
def test_matrix_core_path_beyond_2GiB(nmfk, orc, k):
    # V 600000 x 1000 (2.4 GB, and its transposed copy): both half-steps stream a U larger
    # than a 32-bit byte offset reaches.  The matrix-core path must agree with the
    # vector-ALU path (plain pointers) on the same start.
    n, m = 600000, 1000
    with nmfk.Job(n, m, k) as j:
        j.gen_V_planted(77, 12, 0.3)
        out = {}
        for path in (2, 1):
            j.set_kernel_path(path)
            j.init_random(3)
            r = j.run(6, 3, 1000)
            assert r["iterations"] == 6
            out[path] = (j.get_W(), j.get_H())
    assert rel_err(out[2][0], out[1][0]) < 1e-4 and rel_err(out[2][1], out[1][1]) < 1e-4


def test_transpose_beyond_65535_row_tiles(nmfk, orc):
    # 4.3 million rows: more 64-row tiles than a grid's y extent holds, so the transposed
    # copy of V (the W half's input) is built by tiles strided over the grid.
    # One W half-step (it reads only the transposed copy) against the FP64 oracle.
    n, m, k = 4_300_000, 8, 2
    V = orc.gen_lognormal(n, m, 19, 0.0, 1.0)
    with nmfk.Job(n, m, k) as j:
        j.set_V(V)
        j.init_random(5)
        j.update_W()
        W = j.get_W()
    W0, H0 = orc.init_WH(n, m, k, 5)
    assert rel_err(W, orc.update_W(V, W0, H0)) < 1e-5


# ---------------------------------------------------------------- full-size runs against FP64

@pytest.mark.parametrize("n,m,k", [(20000, 1000, 16), (60000, 500, 16), (8000, 3000, 32)])
def test_replan_to_targets(nmfk, n, m, k):
    # A job's split buffer covers its lone plan and a replan to the default workgroup target,
    # which skips the lone-job rules (2 x 2 waves, balanced splits) and may split more: every
    # target runs, target 0 gives the lone plan back, and the half-steps of the two plans
    # agree within the FP32 bar (their sums run in different orders).
    jobs = [nmfk.Job(n, m, k) for _ in range(2)]
    try:
        for j in jobs:
            j.gen_V_planted(7, 8, 0.3)
            j.init_random(3)
        lone = jobs[0].plan()
        for t in (8, 64, 1024, 0):
            jobs[1].replan(t)
        assert jobs[1].plan() == lone
        jobs[1].replan(1024)
        assert jobs[1].plan()["H"]["S"] >= lone["H"]["S"]
        for j in jobs:
            j.update_H()
            j.update_W()
        assert rel_err(jobs[1].get_H(), jobs[0].get_H()) < 1e-5
        assert rel_err(jobs[1].get_W(), jobs[0].get_W()) < 1e-5
    finally:
        for j in jobs:
            j.close()


def _large_fixture(name):
    f = GOLDEN / f"{name}.npz"
    if not f.exists():
        pytest.skip(f"{f.name} not generated (tests/golden/make_golden.py --large)")
    return np.load(f)


def _device_run_vs_fp64(nmfk, g, path=None, trace=True, sched=0):
    n, m, k, kstar, sv, si, iters, step = (int(x) for x in g["params"])
    with nmfk.Job(n, m, k) as job:
        job.gen_V_planted(sv, kstar, 0.3)
        V = job.get_V()
        # the device generated the oracle's V
        assert float(V.astype(np.float64).sum()) == float(g["V_checksum"])
        assert np.array_equal(V[g["V_probe_idx"], [(i * 104729) % m for i in range(64)]], g["V_probe"])
        del V
        if path is not None:
            job.set_kernel_path(path)
        job.set_schedule(sched)
        job.init_random(si)
        r = job.run(iters, 10, 10**9, trace=trace)
        dv, dvwh, kl = job.dot_kl()
        W, H, cls = job.get_W(), job.get_H(), job.get_classification()
    rows = np.arange(0, n, step)
    WH = W[rows].astype(np.float64) @ H.T.astype(np.float64)
    WHr = g["W_rows"].astype(np.float64) @ g["H"].T.astype(np.float64)
    err = {"rel_kl": abs(kl - float(g["kl"])) / float(g["kl"]),
           "rel_frobenius_WH_sample": float(np.linalg.norm(WH - WHr) / np.linalg.norm(WHr)),
           "rel_H": rel_err(H, g["H"]), "rel_W_sample": rel_err(W[rows], g["W_rows"]),
           "rel_dist": abs(np.sqrt(dvwh / dv) - np.sqrt(float(g["dot_VWH"]) / float(g["dot_V"])))
           / np.sqrt(float(g["dot_VWH"]) / float(g["dot_V"])),
           "class_agreement": float(np.mean(cls == g["cls"]))}
    return r, cls, err


@pytest.mark.parametrize("sched", [2, 1], ids=["one_pass", "two_pass"])
def test_config1_full_run_against_fp64(nmfk, sched):
    # The benchmarked workload itself: V 20000 x 1000 planted rank 16, k = 16, 500 iterations
    # (FP32 matrix cores; one pass per half-step, the default, and one pass over V per
    # iteration), against the FP64 oracle run from the same W0, H0.
    g = _large_fixture("config1_fp64")
    r, cls, err = _device_run_vs_fp64(nmfk, g, sched=sched)
    print(f"config1 FP32 schedule {sched} vs FP64:", err)
    assert r["iterations"] == int(g["iterations"]) and r["ntests"] == int(g["ntests"])
    assert err["rel_kl"] <= 1e-3 and err["rel_dist"] <= 1e-3
    assert err["rel_frobenius_WH_sample"] <= 1e-3
    assert np.array_equal(cls, g["cls"])
    want = g["diff_trace"]
    if sched == 1:
        assert np.array_equal(r["diff_trace"], want)
    else:
        # The one-pass schedule adds its sums in another order: a column whose two largest
        # factors of H tie to within FP32 rounding can take the other class at a test on the
        # way (seen at 2 of the 50 tests), which moves that test's count.  What the stop rule
        # reads, whether a count is zero, must match at every test, and the counts at all but
        # two tests.
        got = r["diff_trace"]
        assert np.array_equal(got == 0, want == 0)
        assert np.count_nonzero(got != want) <= 2, (got, want)


@pytest.mark.parametrize("path", [3, 2], ids=["bf16", "fp32"])
def test_config3_full_run_against_fp64(nmfk, path):
    # Dense rank: V 50000 x 2000 planted rank 48, k = 64, 300 iterations.  BF16 contractions
    # with FP32 accumulation (path 3, the default at k = 64) and FP32 matrix cores (path 2)
    # against FP64.  Stated bounds: KL within 1e-3 relative on both paths; W.H (every 25th
    # row) within 1e-3 relative Frobenius; class vectors: FP32 equal to FP64, BF16 at least
    # 99% equal (its products round the operands to 8 significant bits).
    g = _large_fixture("config3_fp64")
    r, cls, err = _device_run_vs_fp64(nmfk, g, path=path, trace=False)
    print(f"config3 path {path} vs FP64:", err)
    assert r["iterations"] == int(g["iterations"])
    assert err["rel_kl"] <= 1e-3 and err["rel_dist"] <= 1e-3
    assert err["rel_frobenius_WH_sample"] <= 1e-3
    if path == 2:
        assert np.array_equal(cls, g["cls"])
    else:
        assert err["class_agreement"] >= 0.99


@pytest.mark.parametrize("n,m,k,ldv", [(18, 70, 3, 36_000_001), (40, 257, 12, 33_554_433), (5, 9, 2, 150_000_000)])
def test_dot_kl_of_very_long_rows(nmfk, orc, n, m, k, ldv):
    # Rows of V so far apart that 16 of them pass 2 GiB: as right as any other pitch.  V is a few
    # columns of a wider matrix on the device, at the bar of test_dot_and_kl_match_oracle.
    hip = C.CDLL("libamdhip64.so")
    hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    hip.hipFree.argtypes = [C.c_void_p]
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    V = orc.gen_lognormal(n, m, 7, 0.0, 1.0)
    W, H = orc.init_WH(n, m, k, 5)
    dV, out = C.c_void_p(), np.empty(3)
    lib = nmfk.load()
    assert hip.hipMalloc(C.byref(dV), 4 * ((n - 1) * ldv + m) + 64) == 0
    try:
        d_out = C.c_void_p(dV.value + 4 * m // 64 * 64 + 64)   # between the first two rows
        for i in range(n):
            assert hip.hipMemcpy(dV.value + 4 * i * ldv, V[i].ctypes.data, 4 * m, 1) == 0
        with nmfk.Job(n, m, k) as job:
            job.set_WH(W, H)
            inf = job.info()
            job.sync()
            assert lib.nmfk_dot_kl_noalloc(dV, ldv, inf.dW, inf.dH, n, m, k, d_out, inf.stream) == 0, nmfk.last_error()
            job.sync()
        assert hip.hipMemcpy(out.ctypes.data, d_out, 24, 2) == 0
    finally:
        hip.hipFree(dV)
    dv, dvwh = orc.dot_VWH(V.astype(np.float64), W.astype(np.float64), H.astype(np.float64))
    kl = orc.kl_div(V, W, H, fp64=True)
    assert abs(out[0] - dv) / dv < 1e-12 and abs(out[1] - dvwh) / dvwh < 1e-9 and abs(out[2] - kl) / kl < 1e-9


@pytest.mark.parametrize("n,m,k,path", [(2111, 63, 16, 2), (60, 5000, 9, 2), (2111, 63, 48, 3), (5000, 20, 4, 1), (4000, 1500, 12, 2)])
def test_timing_describes_the_launches_of_a_run(nmfk, n, m, k, path):
    # A half-step of one split is one launch, whose finish has no time of its own.
    with nmfk.Job(n, m, k) as job:
        job.set_kernel_path(path)
        job.gen_V_lognormal(3, 0.0, 1.0)
        job.init_random(4)
        t, pl = job.time_iterations(3), job.plan()
        assert t["ms_per_iter"] > 0
        for half in "HW":
            assert t[f"ms_partial_{half}"] > 0 and (t[f"ms_finish_{half}"] == 0) == (pl[half]["S"] == 1)
