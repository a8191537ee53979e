"""GPU parity: the HIP path through the C ABI against the FP64 CPU oracle on the
same inputs.  Integer-valued golden data must match exactly; FP64 runs within
the tolerances written in each test (1e-12 relative for the plain FP64 path's
factors and costs).  ALS runs compare every discrete decision; a line-search test
whose two costs tie to rounding may go either way, so the oracle is run on the
device's line-search outcomes and every sweep where they differ from its own test
must be such a tie -- the final factors are compared in every case.  Full-size
checks use the closed form of an exact low-rank MTTKRP (800^3, 200^4) and a
three-sweep 800^3 ALS against the oracle."""
import os
import sys

import numpy as np
import pytest

import oracle as o
import parity_util as U
import ptn_hip as P

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-test]", *a, flush=True)


@pytest.fixture(scope="module")
def h():
    say("create handle")
    with P.Handle(0) as hd:
        yield hd


# ------------------------------------------------------------------ MTTKRP --

@pytest.mark.parametrize("name", ["mttkrp_3x4x5_r2.npz", "mttkrp_2x3x4x5_r3.npz"])
def test_mttkrp_golden_exact(h, golden_dir, name):
    say("golden", name)
    g = np.load(os.path.join(golden_dir, name))
    dims = [int(d) for d in g["dims"]]
    X = g["X"].reshape(dims, order="F")
    A = [g["A%d" % k] for k in range(len(dims))]
    h.set_tensor(X)
    for mode in range(len(dims)):
        assert np.array_equal(h.mttkrp(A, mode), g["M%d" % mode]), mode
    if len(dims) in (3, 4):
        D = h.mttkrp_dimtree(A)
        for mode in range(len(dims)):
            assert np.array_equal(D[mode], g["M%d" % mode]), mode


@pytest.mark.parametrize("dims,R", [([100, 100, 100], 10), ([37, 23, 41], 5), ([17, 65, 33], 33),
                                    ([64, 16, 48], 64), ([9, 11, 13, 7], 17), ([3, 5, 4, 2, 3], 6),
                                    ([20, 20, 30, 31], 40)])
def test_mttkrp_vs_oracle(h, dims, R):
    """Every mode and form against the oracle; [20, 20, 30, 31] gives the order-4 left node
    three k splits (400 rows, k = 930) whose last ends in a partial 16-k step."""
    say("mttkrp", dims, R)
    rng = np.random.default_rng(sum(dims) + R)
    X = np.asfortranarray(rng.standard_normal(dims))
    A = [rng.random((I, R)) for I in dims]
    h.set_tensor(X, storage=P.TENSOR_BOTH)
    for mode in range(len(dims)):
        ref = o.mttkrp(X, A, mode)
        got = h.mttkrp(A, mode)
        assert P.rel_err(got, ref) < 1e-13, (mode, P.rel_err(got, ref))
        # FP32 tensor stream with FP64 matrix cores: bounded by the FP32 rounding of X
        got32 = h.mttkrp(A, mode, arith=P.ARITH_F32_F64)
        assert P.rel_err(got32, ref) < 1e-6
        # FP32 matrix cores (FP32 products, FP32 accumulation) and bf16x3 split products
        assert P.rel_err(h.mttkrp(A, mode, arith=P.ARITH_F32), ref) < 2e-5, mode
        assert P.rel_err(h.mttkrp(A, mode, arith=P.ARITH_BF16X3), ref) < 2e-4, mode
    if len(dims) in (3, 4):
        D = h.mttkrp_dimtree(A)
        D3 = h.mttkrp_dimtree(A, arith=P.ARITH_BF16X3)
        D2 = h.mttkrp_dimtree(A, arith=P.ARITH_F32)
        for mode in range(len(dims)):
            ref = o.mttkrp(X, A, mode)
            assert P.rel_err(D[mode], ref) < 1e-13, mode
            assert P.rel_err(D2[mode], ref) < 2e-5, mode
            assert P.rel_err(D3[mode], ref) < 2e-4, mode


def test_mttkrp_full_size_closed_form(h):
    """800^3 exact rank-32 tensor: M_n = B_n (Hadamard_{k!=n} B_k^T A_k)."""
    dims, Rt, R = [800, 800, 800], 32, 32
    say("full size closed form", dims)
    h.generate_tensor(dims, Rt, seed=0, snr_db=None, storage=P.TENSOR_BOTH)
    B = o.gen_factors(dims, Rt, seed=0)
    A = o.gen_factors(dims, R, seed=1)
    for mode in range(3):
        H = np.ones((Rt, R))
        for k in range(3):
            if k != mode:
                H *= B[k].T @ A[k]
        ref = B[mode] @ H
        assert P.rel_err(h.mttkrp(A, mode), ref) < 1e-12, mode
    D = h.mttkrp_dimtree(A)
    D3 = h.mttkrp_dimtree(A, arith=P.ARITH_BF16X3)
    D2 = h.mttkrp_dimtree(A, arith=P.ARITH_F32)
    for mode in range(3):
        H = np.ones((Rt, R))
        for k in range(3):
            if k != mode:
                H *= B[k].T @ A[k]
        ref = B[mode] @ H
        assert P.rel_err(D[mode], ref) < 1e-12, mode
        say("full size", mode, "fp32 mfma err", P.rel_err(D2[mode], ref), "bf16x3 err", P.rel_err(D3[mode], ref))
        assert P.rel_err(D2[mode], ref) < 1e-5, mode
        assert P.rel_err(D3[mode], ref) < 1e-4, mode


def test_left_node_over_4gb_k_range_closed_form(h):
    """1100 x 1000 x 1000 FP32 (4.4 GB): the left node's k range spans more than 4 GB, so the
    strided contraction loads through 64-bit addresses instead of a raw buffer; the tree's
    MTTKRPs of the exact rank-8 tensor still match the closed form M_n = B_n (o B_k^T A_k)."""
    dims, Rt, R = [1100, 1000, 1000], 8, 32
    say("left node over a 4 GB k range", dims)
    h.generate_tensor(dims, Rt, seed=0, snr_db=None, storage=P.TENSOR_F32)
    B = o.gen_factors(dims, Rt, seed=0)
    A = o.gen_factors(dims, R, seed=1)
    for ar, tol in ((P.ARITH_F32, 1e-5), (P.ARITH_BF16X3, 1e-4)):
        D = h.mttkrp_dimtree(A, arith=ar)
        for mode in range(3):
            H = np.ones((Rt, R))
            for k in range(3):
                if k != mode:
                    H *= B[k].T @ A[k]
            err = P.rel_err(D[mode], B[mode] @ H)
            say("arith", ar, "mode", mode, "rel err", err)
            assert err < tol, (ar, mode, err)
    h.set_tensor(np.ones((2, 2, 2), order="F"))          # release the 4.4 GB


# --------------------------------------------------------- generator / cost --

def test_generator_matches_oracle(h):
    say("generator")
    dims = [30, 20, 10]
    A_gpu = h.generate_factors(dims, 7, seed=5)
    A_cpu = o.gen_factors(dims, 7, seed=5)
    for a, b in zip(A_gpu, A_cpu):
        assert np.array_equal(a, b)                       # integer arithmetic + exact conversion
    h.generate_tensor(dims, 4, seed=3, snr_db=None)
    X0, _ = o.make_tensor(dims, 4, seed=3)
    assert h.norm_sq() == pytest.approx(np.sum(X0 ** 2), rel=1e-14)
    h.generate_tensor(dims, 4, seed=3, snr_db=20.0)
    Xn, _ = o.make_tensor(dims, 4, seed=3, snr_db=20.0)
    assert h.norm_sq() == pytest.approx(np.sum(Xn ** 2), rel=1e-12)


def test_cost_explicit_matches_oracle(h):
    say("explicit cost")
    X, At = o.make_tensor([40, 30, 20], 5, seed=0, snr_db=25.0)
    init = o.gen_factors([40, 30, 20], 5, seed=1)
    h.set_tensor(X)
    assert h.cost_explicit(init) == pytest.approx(o.cost_explicit(X, init), rel=1e-13)


@pytest.mark.parametrize("storage", [P.TENSOR_F64, P.TENSOR_F32])
@pytest.mark.parametrize("dims,R", [((1, 3, 5), 1), ((16, 8, 8), 16), ((17, 13, 5), 17), ((200, 7, 3), 33),
                                    ((33, 300, 31), 48), ((15, 129, 130), 49), ((31, 9, 10, 7), 64),
                                    ((3, 4, 3, 5, 6), 20), ((700, 64, 33), 5)])
def test_cost_explicit_at_the_tiles_edges(h, dims, R, storage):
    """Rows of mode 0 in tiles of 16, columns in groups of 128 or 256, mode 0 split where columns
    are few, every padded rank, FP64 and FP32 tensors (FP32 values in both), against numpy in
    FP64.  A sum of positive terms of few roundings each: 1e-13 relative."""
    rng = np.random.default_rng(R)
    X = rng.standard_normal(dims).astype(np.float32).astype(np.float64)
    A = [rng.random((I, R)) for I in dims]
    rec = A[0]
    for a in A[1:]:
        rec = rec[..., None, :] * a
    h.set_tensor(X, storage=storage)
    assert h.cost_explicit(A) == pytest.approx(np.linalg.norm(X - rec.sum(-1)), rel=1e-13)


# ------------------------------------------------------------ R x R pieces --

def test_sym_extremes_match_oracle(h, golden_dir):
    g = np.load(os.path.join(golden_dir, "eig_extremes.npz"))
    for i in range(int(g["count"])):
        V = g["V%d" % i]
        say("eig", V.shape)
        L, mu = h.sym_extremes(V)
        Lo, muo, _ = o.sym_extremes(V)
        assert L == Lo and mu == muo                       # same arithmetic sequence: bitwise


@pytest.mark.parametrize("n,kind", [(1, "scalar"), (2, "pair"), (7, "indefinite"), (17, "indefinite"),
                                    (33, "indefinite"), (64, "indefinite"), (20, "negdef"), (64, "psd_rankdef"),
                                    (9, "diag"), (40, "blockdiag")])
def test_sym_extremes_edge_cases_match_oracle(h, n, kind):
    """Spectra the Nesterov constants rarely see: eigenvalues of both signs (the pair
    bracketed around 0), all negative, rank-deficient, and matrices with zero columns to
    eliminate (the no-reflection branch), at every padded size (16, 32, 64): bitwise."""
    say("eig edge", n, kind)
    rng = np.random.default_rng(100 + n)
    if kind in ("scalar", "pair", "indefinite"):
        B = rng.standard_normal((n, n))
        V = 0.5 * (B + B.T)
    elif kind == "negdef":
        B = rng.random((n, 2 * n))
        V = -(B @ B.T)
    elif kind == "psd_rankdef":
        B = rng.random((n, n // 2))
        V = B @ B.T
    elif kind == "diag":
        V = np.diag(rng.standard_normal(n))
    else:                                                  # two blocks: zero entries below the first
        V = np.zeros((n, n))
        for a, b in ((0, n // 2), (n // 2, n)):
            B = rng.standard_normal((b - a, b - a))
            V[a:b, a:b] = 0.5 * (B + B.T)
    L, mu = h.sym_extremes(V)
    Lo, muo, _ = o.sym_extremes(V)
    assert L == Lo and mu == muo


@pytest.mark.parametrize("R", [1, 2, 3, 4, 5, 15, 16, 17, 18, 31, 32, 33, 61, 63, 64])
def test_extremes_at_the_edges_of_the_padded_ranks(h, R):
    # bitwise the oracle's on both sides of the routine's forms (one wave, two, four; pivot
    # steps in fours): plain, indefinite, and what its branches look for, uncoupled columns
    # (a column to eliminate that is zero already), repeated and zero eigenvalues, and entries
    # whose squares leave the range in which the short division is taken
    rng = np.random.default_rng(R)
    B = rng.standard_normal((2 * R + 1, R))
    S = rng.standard_normal((R, R))
    D = np.diag(rng.standard_normal(R))
    K = np.kron(np.eye((R + 2) // 3), np.ones((3, 3)))[:R, :R]
    for name, V in (("gram", B.T @ B), ("indefinite", S + S.T), ("diagonal", D), ("blocks", K), ("ones", np.ones((R, R))),
                    ("zero", np.zeros((R, R))), ("identity", np.eye(R)), ("large", (B.T @ B) * 2.0**300),
                    ("small", (S + S.T) * 2.0**-300), ("graded", (B.T @ B) * np.outer(*[10.0 ** -np.arange(R)] * 2))):
        V = (V + V.T) / 2
        L, mu = h.sym_extremes(V)
        Lo, muo, _ = o.sym_extremes(V)
        assert L == Lo and mu == muo, name


@pytest.mark.parametrize("I,R,d", [(7, 4, 1e-2), (300, 32, 1e-2), (129, 64, 1e-2), (50, 10, 0.0), (20, 5, 1e30)])
def test_nesterov_matches_oracle(h, I, R, d):
    say("nnls", I, R, d)
    rng = np.random.default_rng(I + R)
    B = rng.random((3 * R, R))
    Z = B.T @ B
    W = rng.standard_normal((I, R)) * 4 + 2
    A0 = rng.random((I, R))
    Ag, itg, Lg, mug = h.nesterov(Z, W, A0, d, d, 50)
    Ao, ito, Lo, muo, = o.nesterov(Z, W, A0, d, d, 50)
    assert itg == ito
    assert (Lg, mug) == (Lo, muo)
    assert np.array_equal(Ag, Ao)                          # row arithmetic mirrors the oracle


@pytest.mark.parametrize("R", [1, 2, 3, 15, 16, 17, 31, 32, 33])
def test_nesterov_at_the_edges_of_the_padded_ranks(h, R):
    # bitwise the oracle's where a wave holds one, two and four copies of a row
    rng = np.random.default_rng(60 + R)
    B = rng.random((3 * R, R))
    for I in (1, 5):
        W = rng.standard_normal((I, R)) * 4 + 2
        A0 = rng.random((I, R))
        Ag, itg, Lg, mug = h.nesterov(B.T @ B, W, A0, 1e-2, 1e-2, 70)
        Ao, ito, Lo, muo = o.nesterov(B.T @ B, W, A0, 1e-2, 1e-2, 70)
        assert itg == ito and (Lg, mug) == (Lo, muo)
        assert np.array_equal(Ag, Ao)


@pytest.mark.parametrize("wf", [0, 1, 2, 3])
def test_normalize_matches_oracle(h, wf):
    """Normalize with the weights loaded on factor wf (Normalize.hpp:92-174): bitwise the
    oracle's, including the zero-norm branch, for every weight factor of orders 3 and 4."""
    rng = np.random.default_rng(3 + wf)
    for N in (3, 4):
        if wf >= N:
            continue
        dims = [7, 6, 5, 4][:N]
        A = [rng.random((I, 5)) for I in dims]
        A[-1][:, 2] = 0.0                                  # zero-norm branch on one column
        A[N - 2][:, 4] = 0.0                               # ... the one wf = N - 1 reads
        G = [a.T @ a for a in A]
        say("normalize N=%d wf=%d" % (N, wf))
        Gg, Ag = h.normalize(G, A, wf)
        Go, Ao = o.normalize(G, A, wf)
        for a, b in zip(Ag, Ao):           # a zero norm the test does not read divides by 0: NaN on both
            assert np.array_equal(a, b, equal_nan=True)
        for a, b in zip(Gg, Go):
            assert np.array_equal(a, b, equal_nan=True)


def test_order4_gemm_node_full_size_closed_form(h):
    """200^4 (6.4 GB FP32, 12.8 GB FP64), noiseless and of exact rank 64 with Exponential(1)
    factors: every MTTKRP of the tree -- the order-4 GEMM node in FP32 MFMA and bf16x3, and
    the FP64 path on the FP64 copy -- against the closed form M_n = B_n (o_{k!=n} B_k^T A_k).
    Tolerances: FP64 1e-12; FP32 rounding of X plus FP32 accumulation over k = 40000 in
    split chunks 1e-5 (FP32 MFMA) and 1e-4 (bf16x3)."""
    dims, Rt, R = [200, 200, 200, 200], 64, 64
    say("order-4 node 200^4 R=64 closed form")
    h.generate_tensor(dims, Rt, seed=2, snr_db=None, dist=1, storage=P.TENSOR_BOTH)
    B = o.gen_factors(dims, Rt, seed=2, dist=1)
    A = h.generate_factors(dims, R, seed=1)
    refs = []
    for mode in range(4):
        H = np.ones((Rt, R))
        for k in range(4):
            if k != mode:
                H *= B[k].T @ A[k]
        refs.append(B[mode] @ H)
    for ar, tol in ((P.ARITH_F64, 1e-12), (P.ARITH_F32, 1e-5), (P.ARITH_BF16X3, 1e-4)):
        M = h.mttkrp_dimtree(A, arith=ar)
        errs = [P.rel_err(M[k], refs[k]) for k in range(4)]
        say("arith", ar, "rel errs vs closed form", ["%.2e" % e for e in errs])
        assert max(errs) < tol, (ar, errs)
    h.set_tensor(np.ones((2, 2, 2), order="F"))          # release the 19 GB


# --------------------------------------------------------------------- ALS --

TOL = 1e-12       # plain FP64 path: factors, relative
COST_TOL = 2e-13  # |f_device^2 - f_oracle^2| / ||X||^2 (see _compare_runs)
TIE = 1e-12       # |f - f_accel| / f below which a line-search outcome rests on rounding


def oracle_on_device_path(X, R, init, logg, tie=TIE, **kw):
    return U.oracle_on_device_path(X, R, init, logg, tie, **kw)


def _compare_runs(Fg, stg, logg, Fo, sto, logo, tol=TOL, cost_tol=COST_TOL):
    """Every discrete decision equal; factors within tol.  Costs are compared on the scale
    of ||X||^2: the Gram-form cost f^2 = ||X||^2 - 2<M, A> + <V, G> is a difference of
    three terms of that size, each a sum of up to 10^6 products taken in another order on
    each side (the oracle sums ||X||^2 sequentially in chunks of 65 536, ~sqrt(65536) eps =
    3e-14 of rounding), so f^2 agrees to COST_TOL of ||X||^2 (measured <= 2.2e-14 here,
    6.5e-14 in the batch tests), which near the noise floor is ~1e-12 of f itself."""
    assert stg["ao_iter"] == sto["ao_iter"]
    assert [l["nnls_iters"] for l in logg] == [l["nnls_iters"] for l in logo]
    assert [l["accel_tried"] for l in logg] == [l["accel_tried"] for l in logo]
    assert [l["accel_accepted"] for l in logg] == [l["accel_accepted"] for l in logo]
    assert [l["zero_col_fallback"] for l in logg] == [l["zero_col_fallback"] for l in logo]
    frob = sto["frob_sq"]
    fgap = max(abs(a["f_value"] ** 2 - b["f_value"] ** 2) for a, b in zip(logg, logo)) / frob
    agap = max([abs(a["f_accel"] ** 2 - b["f_accel"] ** 2) for a, b in zip(logg, logo) if b["accel_tried"]]
               or [0.0]) / frob
    ferr = max(P.rel_err(a, b) for a, b in zip(Fg, Fo))
    say("vs oracle: final factors %.2e (tolerance %.1e); max |f^2 - f_o^2| / ||X||^2 %.2e, accelerated %.2e "
        "(tolerance %.1e)" % (ferr, tol, fgap, agap, cost_tol))
    assert fgap < cost_tol and agap < cost_tol
    assert (stg["accel_coeff"], stg["accel_fail"]) == (sto["accel_coeff"], sto["accel_fail"])
    assert ferr < tol


def _als_parity(h, X, R, init, oform=o.MTTKRP_STANDARD, **kw):
    """One device run through the C ABI against the oracle's run on its path.  The factor
    (cost) tolerance is 1e-12 (COST_TOL), or four times the spread between the oracle's own
    summation orders (per-mode, blocked and tree MTTKRP on the same path) where the problem
    amplifies rounding beyond that: the orthogonality branch's (M^T M)^-1/2 and the
    unconstrained M V^-1 reach a 2.5e-11 spread after ten sweeps in the oracle alone."""
    Fg, stg, logg = h.cpd(R, init, **kw)
    okw = {k: v for k, v in kw.items() if k != "mttkrp_form"}
    Fo, sto, logo = oracle_on_device_path(X, R, init, logg, mttkrp_form=oform, cost_form=o.COST_GRAM, **okw)
    spread, cspread = U.oracle_spread(X, R, init, logg, Fo, logo, oform, cost_form=o.COST_GRAM, **okw)
    say("oracle's own spread between summation orders: factors %.2e, |f^2 - f^2| / ||X||^2 %.2e"
        % (spread, cspread))
    _compare_runs(Fg, stg, logg, Fo, sto, logo, max(TOL, 4.0 * spread), max(COST_TOL, 4.0 * cspread))
    return Fg, stg, logg


def _oform(form):
    return o.MTTKRP_DIMTREE if form == P.MTTKRP_DIMTREE else o.MTTKRP_STANDARD


@pytest.mark.parametrize("form", [P.MTTKRP_STANDARD, P.MTTKRP_DIMTREE])
def test_als_c1_parity(h, form):
    """Config 1: 100^3, R=10, SNR 30 dB, init seed 1, 50 sweeps, reference defaults."""
    say("ALS C1 form", form)
    dims, R = [100, 100, 100], 10
    X, _ = o.make_tensor(dims, R, seed=0, snr_db=30.0)
    init = o.gen_factors(dims, R, seed=1)
    h.set_tensor(X)
    Fg, stg, logg = _als_parity(h, X, R, init, mttkrp_form=form, oform=_oform(form), max_iter=50,
                                threshold_error=0.0)
    say("rel", stg["rel_cost"], "sweeps/s", stg["ao_iter"] / stg["sweep_seconds"])


@pytest.mark.parametrize("form", [P.MTTKRP_STANDARD, P.MTTKRP_DIMTREE])
def test_als_threshold_stop(h, form):
    """The relative-cost threshold ends the run at the same sweep as the oracle; the
    stopping sweep takes no acceleration step (termination precedes line_search_accel)."""
    dims, R = [60, 50, 40], 6
    X, _ = o.make_tensor(dims, R, seed=8, snr_db=30.0)
    init = o.gen_factors(dims, R, seed=9)
    h.set_tensor(X)
    Fg, stg, logg = _als_parity(h, X, R, init, mttkrp_form=form, oform=_oform(form), max_iter=200,
                                threshold_error=0.05)
    say("threshold stop at", stg["ao_iter"])
    assert 1 < stg["ao_iter"] < 200
    assert logg[stg["ao_iter"] - 1]["accel_tried"] == 0


def test_als_c1_no_accel_no_norm(h):
    say("ALS C1 variant: acceleration and normalization off")
    dims, R = [100, 100, 100], 10
    X, _ = o.make_tensor(dims, R, seed=0, snr_db=30.0)
    init = o.gen_factors(dims, R, seed=1)
    h.set_tensor(X)
    _als_parity(h, X, R, init, max_iter=50, threshold_error=0.0, acceleration=0, normalization=0)


@pytest.mark.parametrize("dims,R", [([12, 9, 10, 8], 4), ([30, 31, 32], 33)])
def test_als_small_parity(h, dims, R):
    say("ALS small", dims, R)
    X, _ = o.make_tensor(dims, min(R, 6), seed=2, snr_db=25.0)
    init = o.gen_factors(dims, R, seed=3)
    h.set_tensor(X)
    for form in (P.MTTKRP_STANDARD, P.MTTKRP_DIMTREE):
        _als_parity(h, X, R, init, mttkrp_form=form, oform=_oform(form), max_iter=15, threshold_error=0.0)


@pytest.mark.parametrize("dims,R", [([40, 30, 20], 16), ([40, 30, 20], 17), ([13, 9, 10, 8], 17),
                                    ([128, 128, 64], 32), ([128, 128, 65], 32)])
def test_als_on_one_stream_and_on_two(h, dims, R):
    """Both sides of the rule that keeps a sweep on one stream: the padded rank 16, order 3 and 4 at
    rank 17, and 8 MB of an order-3 tensor at rank 32."""
    X, _ = o.make_tensor(dims, 6, seed=12, snr_db=25.0)
    init = o.gen_factors(dims, R, seed=13)
    h.set_tensor(X)
    for form in (P.MTTKRP_STANDARD, P.MTTKRP_DIMTREE):
        _als_parity(h, X, R, init, mttkrp_form=form, oform=_oform(form), max_iter=6, threshold_error=0.0)


@pytest.mark.parametrize("arith", [P.ARITH_F32, P.ARITH_BF16X3])
@pytest.mark.parametrize("dims,R,cons", [
    ([40, 30, 20], 16, [1, 1, 1]), ([30, 25, 20, 12], 16, [1, 1, 1, 1]),        # one stream
    ([40, 30, 20], 17, [1, 1, 1]), ([13, 9, 10, 8], 17, [1, 1, 1, 1]),          # the contraction aside
    ([45, 40, 30, 20], 33, [1, 1, 1, 1]), ([8, 7, 9, 6, 5], 24, [1, 1, 1, 1, 1]),
    ([175, 170, 160], 10, [1, 1, 1]), ([60, 55, 50, 45], 12, [1, 1, 1, 1]),     # the set-up aside (standard form)
    ([24, 22, 20, 18, 10], 20, [1, 1, 1, 1, 1]),
    ([60, 50, 40], 5, [1, 2, 0]), ([60, 50, 40], 20, [0, 1, 2]), ([24, 20, 22, 26], 20, [1, 0, 1, 2])])
def test_als_fp32_products_on_every_schedule(h, arith, dims, R, cons):
    """FP32 and BF16x3 contractions on each schedule of a sweep (all on one stream, the contraction
    aside, the set-up aside), in both forms, fused and unfused, with mixed constraints.  Against the
    FP64 oracle on the run's own line-search path: FP32 accumulation puts about 1e-6 of ||X||^2 into
    the fit term of f^2 (1e-5 allowed), a hundred times that where unconstrained factors of large
    norm cancel (1e-4).  A second run gives the same bits: nothing read early or late."""
    say("FP32 schedules", dims, R, cons, "arith", arith)
    nonneg = all(c == 1 for c in cons)
    X, _ = o.make_tensor(dims, 5, seed=30, snr_db=25.0)
    init = o.gen_factors(dims, R, seed=31)
    h.set_tensor(X, storage=P.TENSOR_F32)
    frob = float(np.sum(X * X))
    kw = dict(max_iter=4, threshold_error=0.0, constraints=cons)
    for form, fuse in ((P.MTTKRP_STANDARD, 0), (P.MTTKRP_DIMTREE, 0), (P.MTTKRP_DIMTREE, 1)):
        Fg, _, lg = h.cpd(R, init, arith=arith, mttkrp_form=form, fuse_accel=fuse, **kw)
        oform = _oform(form) if len(dims) <= 4 else o.MTTKRP_STANDARD     # (the oracle's tree ends at order 4)
        _, _, logo = oracle_on_device_path(X, R, init, lg, tie=1e-3, mttkrp_form=oform, cost_form=o.COST_GRAM, **kw)
        worst = max(abs(a["f_value"] ** 2 - b["f_value"] ** 2) for a, b in zip(lg, logo)) / frob
        say("form", form, "fused", fuse, "max |f^2 - f_oracle^2| / ||X||^2 = %.2e" % worst)
        assert worst < (1e-5 if nonneg else 1e-4)
        Fa, _, la = h.cpd(R, init, arith=arith, mttkrp_form=form, fuse_accel=fuse, **kw)
        assert [(l["f_value"], l["f_accel"], l["nnls_iters"]) for l in la] == \
            [(l["f_value"], l["f_accel"], l["nnls_iters"]) for l in lg]
        for a, b in zip(Fa, Fg):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("arith", [P.ARITH_F32, P.ARITH_BF16X3])
def test_als_paired_pass_of_order_4_beside_the_set_up(h, arith):
    """The paired line-search pass at order 4 and rank > 16 on a tensor too large for the contraction to
    go aside (297 MB in FP32, over the tree's 288): fused and unfused runs take the same steps and
    agree in every bit while they do."""
    dims, R = [98, 96, 92, 90], 20
    h.generate_tensor(dims, R, seed=8, snr_db=20.0, storage=P.TENSOR_F32)
    init = o.gen_factors(dims, R, seed=9)
    kw = dict(max_iter=4, threshold_error=0.0, mttkrp_form=P.MTTKRP_DIMTREE, arith=arith)
    F0, st0, lg0 = h.cpd(R, init, fuse_accel=0, **kw)
    F1, st1, lg1 = h.cpd(R, init, fuse_accel=1, **kw)
    acc0, acc1 = [l["accel_accepted"] for l in lg0], [l["accel_accepted"] for l in lg1]
    say("accept unfused", acc0, "fused", acc1)
    assert [l["accel_tried"] for l in lg0] == [l["accel_tried"] for l in lg1] and any(l["accel_tried"] for l in lg0)
    same = next((i for i, (a, b) in enumerate(zip(acc0, acc1)) if a != b), len(acc0))
    for a, b in list(zip(lg0, lg1))[:same + 1]:
        assert (a["f_value"], a["nnls_iters"]) == (b["f_value"], b["nnls_iters"])
    if acc0 == acc1:
        for a, b in zip(F0, F1):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("dims,R", [([17, 17, 16, 17, 16], 24), ([20, 18, 18, 18, 16], 16), ([8, 7, 7, 8, 7, 6], 16),
                                    ([66, 62, 60, 40], 20)])
def test_als_fp64_set_up_aside_at_higher_orders(h, dims, R):
    """FP64 standard-form runs of orders 4 to 6 on each schedule: the contraction aside (9.6 MB of order 5 at
    rank 24), the set-up aside (75 MB of order 4 at rank 20), one stream (orders 5 and 6 at rank 16)."""
    X, _ = o.make_tensor(dims, 5, seed=32, snr_db=25.0)
    init = o.gen_factors(dims, R, seed=33)
    h.set_tensor(X)
    _als_parity(h, X, R, init, mttkrp_form=P.MTTKRP_STANDARD, max_iter=4, threshold_error=0.0)


@pytest.mark.parametrize("I0", [1, 64, 65, 300])
@pytest.mark.parametrize("K", [(1, 31), (4, 8), (3, 11), (30, 17), (32, 16), (27, 19), (90, 91)])
def test_mode0_splits(h, I0, K):
    """The FP64 contraction of mode 0 about its splits: one (under 64 columns), under and from sixteen
    (summed in runs), and as many as the rows' blocks leave.  Up to 8190 terms to a sum, each
    side in its own order: 8190 x 2^-53 = 9e-13 at most."""
    rng = np.random.default_rng(I0 + K[0])
    dims = [I0, *K]
    X = rng.random(dims)
    h.set_tensor(X, storage=P.TENSOR_BOTH)
    for R in (5, 33):
        A = [rng.random((d, R)) for d in dims]
        M = o.mttkrp(X, A, 0)
        assert P.rel_err(h.mttkrp(A, 0), M) <= 1e-12
        X32 = X.astype(np.float32).astype(np.float64)
        assert P.rel_err(h.mttkrp(A, 0, arith=P.ARITH_F32_F64), o.mttkrp(X32, A, 0)) <= 1e-12


@pytest.mark.parametrize("dims", [(512, 512, 128), (512, 512, 129), (16, 1448, 1500), (257, 256, 511)])
def test_fp64_column_contraction_at_the_cache_size(h, dims):
    """Mode 0 and the left node on both sides of 256 MB, where FP64 columns of whole cache lines go over to
    non-temporal loads.  X = [[B]] from the library's generator, so M_n = B_n (Hadamard of B_k^T A_k):
    sums of up to 2.2 million positive terms in FP64, about 2e6^0.5 roundings: 1e-12."""
    R = 17
    h.generate_tensor(list(dims), 3, seed=5, storage=P.TENSOR_F64)
    B = o.gen_factors(list(dims), 3, seed=5)
    rng = np.random.default_rng(3)
    A = [rng.random((I, R)) for I in dims]
    want = [B[n] @ np.prod([B[k].T @ A[k] for k in range(3) if k != n], axis=0) for n in range(3)]
    assert P.rel_err(h.mttkrp(A, 0), want[0]) <= 1e-12
    for got, w in zip(h.mttkrp_dimtree(A), want):
        assert P.rel_err(got, w) <= 1e-12


@pytest.mark.parametrize("dims", [[5, 1, 7, 3], [4, 2, 1, 9], [3, 1, 1, 1], [6, 17, 5, 2], [2, 3, 40, 33], [9, 64, 3, 70]])
@pytest.mark.parametrize("R", [3, 16, 17, 33, 64])
def test_order4_leaf_contractions(h, dims, R):
    """The row contraction with two other modes about its groups of rows: single and short modes,
    fewer rows than groups, remainders of four.  FP64 sums of at most 4480 x 9 positive terms in
    either order (1e-12), FP32 products over a mode of at most 9 (9 x 2^-23 and the data's rounding)."""
    rng = np.random.default_rng(R + dims[1])
    X = rng.random(dims)
    A = [rng.random((d, R)) for d in dims]
    h.set_tensor(X, storage=P.TENSOR_BOTH)
    for mode in (1, 2, 3):
        M = o.mttkrp(X, A, mode)
        assert P.rel_err(h.mttkrp(A, mode), M) <= 1e-12
        assert P.rel_err(h.mttkrp(A, mode, arith=P.ARITH_F32), M) <= 2e-6


@pytest.mark.parametrize("dims", [[3, 1, 1], [3, 7, 512], [3, 7, 513], [3, 513, 7], [2, 255, 300], [2, 256, 300],
                                  [2, 300, 257], [5, 64, 65]])
@pytest.mark.parametrize("R", [1, 16, 17, 48, 64])
def test_leaf_contractions_a_block_to_a_row(h, dims, R):
    """Order 3, modes 1 and 2: both sides of the rule that gives an FP64 node's output row a block of
    its own, fewer rows than groups of threads and remainders of their fours.  At most 513 x 5
    positive FP64 terms in either order (1e-12)."""
    rng = np.random.default_rng(R + dims[2])
    X = rng.random(dims)
    A = [rng.random((d, R)) for d in dims]
    h.set_tensor(X)
    for mode in (1, 2):
        assert P.rel_err(h.mttkrp(A, mode), o.mttkrp(X, A, mode)) <= 1e-12
    for a, b in zip(h.mttkrp_dimtree(A), [o.mttkrp(X, A, m) for m in range(3)]):
        assert P.rel_err(a, b) <= 1e-12


def test_als_c2_full_size_three_sweeps(h):
    """Config 2 at full size (800^3, true rank 32, SNR 20 dB, R = 32, init seed 1): three
    sweeps (the line search runs at sweep 2) of the plain FP64 path, per-mode and tree, against
    the oracle (OpenMP blocked MTTKRP, Gram-form cost) at 1e-12; the FP32-stream forms (tree,
    FP32 MFMA and bf16x3 with the fused line-search pass) end within 1e-6 of the oracle's
    relative error.  The device generates the tensor (bitwise the oracle's generator, tested
    above); its ||X||^2 is checked against the oracle's tensor."""
    dims, R, sweeps = [800, 800, 800], 32, 3
    say("C2 full size: oracle tensor")
    X, _ = o.make_tensor(dims, R, seed=0, snr_db=20.0)
    init = o.gen_factors(dims, R, seed=1)
    say("C2 full size: device tensor")
    h.generate_tensor(dims, R, seed=0, snr_db=20.0, storage=P.TENSOR_BOTH)
    assert h.norm_sq() == pytest.approx(float(np.sum(X * X)), rel=1e-12)
    kw = dict(max_iter=sweeps, threshold_error=0.0)
    say("C2 full size: oracle run")
    Fo, sto, logo = o.cpd(X, R, init, mttkrp_form=o.MTTKRP_BLOCKED, cost_form=o.COST_GRAM, threads=0, **kw)
    assert logo[1]["accel_tried"] == 1
    for form in (P.MTTKRP_STANDARD, P.MTTKRP_DIMTREE):
        say("C2 full size: FP64 form", form)
        Fg, stg, logg = h.cpd(R, init, mttkrp_form=form, **kw)
        assert [l["accel_accepted"] for l in logg] == [l["accel_accepted"] for l in logo]
        _compare_runs(Fg, stg, logg, Fo, sto, logo)
    for ar in (P.ARITH_F32, P.ARITH_BF16X3):
        Fc, stc, _ = h.cpd(R, init, mttkrp_form=P.MTTKRP_DIMTREE, arith=ar, fuse_accel=1, **kw)
        gap = abs(stc["rel_cost"] - sto["rel_cost"])
        ferr = max(P.rel_err(a, b) for a, b in zip(Fc, Fo))
        say("C2 full size: arith", ar, "rel error %.10f vs oracle %.10f (gap %.2e), factors %.2e"
            % (stc["rel_cost"], sto["rel_cost"], gap, ferr))
        assert gap < 1e-6
    h.set_tensor(np.ones((2, 2, 2), order="F"))          # release the 6 GB


@pytest.mark.parametrize("arith", [P.ARITH_F32, P.ARITH_BF16X3])
@pytest.mark.parametrize("dims,R", [([100, 100, 100], 10), ([24, 20, 18, 16], 7)])
def test_als_fp32_stream_and_fused_line_search(h, arith, dims, R):
    """FP32 tensor stream on the dimension tree, with and without the line-search pass
    fused into the next left node.  The paired pass computes the lower half of its
    output column by column exactly as the single left node does, so while the two runs
    take the same acceleration decisions they are bitwise equal apart from f_accel
    (whose fit term is summed in another order).  Against the FP64 oracle the final fit
    agrees to the FP32 stream's accuracy."""
    say("ALS fp32 stream", dims, R, "arith", arith)
    X, _ = o.make_tensor(dims, R, seed=0, snr_db=30.0)
    init = o.gen_factors(dims, R, seed=1)
    h.set_tensor(X, storage=P.TENSOR_BOTH)
    kw = dict(max_iter=25, threshold_error=0.0, mttkrp_form=P.MTTKRP_DIMTREE, arith=arith)
    F0, st0, lg0 = h.cpd(R, init, fuse_accel=0, **kw)
    F1, st1, lg1 = h.cpd(R, init, fuse_accel=1, **kw)
    acc0 = [l["accel_accepted"] for l in lg0]
    acc1 = [l["accel_accepted"] for l in lg1]
    say("accept unfused", acc0, "fused", acc1)
    tried = [i for i, l in enumerate(lg0) if l["accel_tried"]]
    assert tried and [i for i, l in enumerate(lg1) if l["accel_tried"]] == tried
    # first line search: same state in both runs, the fit term <X, [[Ahat]]> summed in
    # another order; FP32 accumulation bounds its difference by ~1e-6 of ||X||^2
    frob = float(np.sum(X * X))
    i = tried[0]
    fa0, fa1 = lg0[i]["f_accel"], lg1[i]["f_accel"]
    say("first f_accel", fa0, fa1, "||X||^2", frob)
    assert abs(fa1 * fa1 - fa0 * fa0) < 1e-5 * frob
    if acc0 == acc1:
        assert [l["nnls_iters"] for l in lg0] == [l["nnls_iters"] for l in lg1]
        for a, b in zip(F0, F1):
            assert np.array_equal(a, b)
    # against the FP64 oracle on each run's own line-search path: FP32 errors scale with
    # ||X||^2 (the fit term <M, A> carries ~1e-7 of it), so squared residuals are compared on
    # that scale, and a line-search outcome is a tie when the oracle's two costs are within
    # the ~1e-4 relative error this puts on f (1e-3 allowed)
    rel_o = None
    for F, lg in ((F0, lg0), (F1, lg1)):
        Fo, sto, logo = oracle_on_device_path(X, R, init, lg, tie=1e-3, mttkrp_form=o.MTTKRP_DIMTREE,
                                              cost_form=o.COST_GRAM, max_iter=25, threshold_error=0.0)
        worst = max(abs(a["f_value"] ** 2 - b["f_value"] ** 2) for a, b in zip(lg, logo)) / frob
        rel = h.cost_explicit(F) / np.sqrt(frob)
        rel_o = o.cost_explicit(X, Fo) / np.sqrt(frob)
        say("on the device's path: max |f^2 - f_oracle^2| / ||X||^2 = %.2e; final rel cost %.10f, oracle %.10f"
            % (worst, rel, rel_o))
        assert worst < 1e-5
        assert abs(rel * rel - rel_o * rel_o) < 1e-5


def test_time_passes_events_leave_results_unchanged(h):
    """time_passes brackets the two tensor passes of every sweep with HIP events: the
    factors, costs and decisions are bitwise those of the untimed run, the order-3 tree
    reports both passes in every sweep that runs them (the left-node pass from sweep 1, the
    paired one from the line search on; the right-node pass in every sweep), and the
    per-sweep times stay within that sweep's wall time."""
    dims, R = [120, 110, 100], 12
    X, _ = o.make_tensor(dims, R, seed=4, snr_db=30.0)
    init = o.gen_factors(dims, R, seed=5)
    h.set_tensor(X, storage=P.TENSOR_F32)
    kw = dict(max_iter=10, threshold_error=0.0, mttkrp_form=P.MTTKRP_DIMTREE, arith=P.ARITH_BF16X3, fuse_accel=1)
    F0, st0, lg0 = h.cpd(R, init, **kw)
    F1, st1, lg1 = h.cpd(R, init, time_passes=1, **kw)
    assert st0["f_value"] == st1["f_value"]
    assert [l["f_accel"] for l in lg0] == [l["f_accel"] for l in lg1]
    for a, b in zip(F0, F1):
        assert np.array_equal(a, b)
    assert all(l["t_pass_ms"] == [0.0, 0.0] for l in lg0)
    t_prev = 0.0
    for k, l in enumerate(lg1):
        left, right = l["t_pass_ms"]
        say("sweep", k + 1, "passes (ms)", left, right)
        assert right > 0.0
        if k + 1 < len(lg1):                 # the last sweep launches no further left-node pass
            assert left > 0.0
        assert left + right < 1e3 * (l["t_end"] - t_prev) + 1.0
        t_prev = l["t_end"]


@pytest.mark.parametrize("R", [3, 16])
@pytest.mark.parametrize("arith", [P.ARITH_F64, P.ARITH_F32_F64])
def test_time_passes_fp64_leaves_results_unchanged(h, arith, R):
    """FP64 contractions of rank <= 16 take the NNLS set-up along as one of their blocks, timed ones
    do not: the same operations in either place, so the same bits."""
    dims = [60, 45, 50]
    X, _ = o.make_tensor(dims, R, seed=4, snr_db=30.0)
    init = o.gen_factors(dims, R, seed=5)
    h.set_tensor(X, storage=P.TENSOR_BOTH)
    for form in (P.MTTKRP_STANDARD, P.MTTKRP_DIMTREE):
        kw = dict(max_iter=8, threshold_error=0.0, mttkrp_form=form, arith=arith)
        F0, st0, lg0 = h.cpd(R, init, **kw)
        F1, st1, lg1 = h.cpd(R, init, time_passes=1, **kw)
        assert st0["f_value"] == st1["f_value"]
        assert [(l["f_value"], l["f_accel"], l["lipschitz"], l["mu"]) for l in lg0] == \
            [(l["f_value"], l["f_accel"], l["lipschitz"], l["mu"]) for l in lg1]
        for a, b in zip(F0, F1):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("dims,R,seed,sweeps", [([5, 4, 6, 3, 4], 3, 5, 9), ([4, 3, 5, 3, 4, 2], 3, 6, 10),
                                                ([3, 4, 5, 3, 2, 3], 2, 7, 10)])
def test_als_higher_order_standard_form(h, dims, R, seed, sweeps):
    """Orders 5 and 6 through the per-mode form."""
    say("ALS order", len(dims), dims, R)
    X, _ = o.make_tensor(dims, R, seed=seed, snr_db=25.0)
    init = o.gen_factors(dims, R, seed=seed + 1)
    h.set_tensor(X)
    _als_parity(h, X, R, init, max_iter=sweeps, threshold_error=0.0)


def _fused_equals_unfused(h, R, init, kw):
    """The tree with FP32 contractions, with and without the line-search pass fused into
    the next left node: while the two runs take the same acceleration decisions they are
    bitwise equal apart from f_accel (its fit term is summed in another order)."""
    kt = dict(kw, mttkrp_form=P.MTTKRP_DIMTREE, arith=P.ARITH_F32)
    F0, st0, lg0 = h.cpd(R, init, fuse_accel=0, **kt)
    F1, st1, lg1 = h.cpd(R, init, fuse_accel=1, **kt)
    acc0 = [l["accel_accepted"] for l in lg0]
    acc1 = [l["accel_accepted"] for l in lg1]
    assert [l["accel_tried"] for l in lg0] == [l["accel_tried"] for l in lg1]
    say("fused line search: accept unfused", acc0, "fused", acc1)
    if acc0 == acc1:
        assert [l["nnls_iters"] for l in lg0] == [l["nnls_iters"] for l in lg1]
        assert st0["f_value"] == st1["f_value"]
        for a, b in zip(F0, F1):
            assert np.array_equal(a, b)
    else:
        k = next(i for i, (a, b) in enumerate(zip(acc0, acc1)) if a != b)
        assert abs(lg0[k]["f_value"] - lg0[k]["f_accel"]) <= 1e-6 * lg0[k]["f_value"], k


@pytest.mark.parametrize("cons", [[0, 0, 0], [2, 1, 1], [1, 0, 2], [1, 4, 1], [0, 2, 1, 3]])
def test_als_other_constraints(h, cons):
    """update_factor's other branches on the device (Cpd.hpp:189-228): unconstrained
    M V^-1 (LU with partial pivoting), orthogonality M (M^T M)^-1/2 (round-robin Jacobi),
    sparsity / constant (factor not updated), mixed with nonnegativity, both MTTKRP forms,
    against the oracle's update_factor; Normalize takes the first non-orthogonal factor."""
    dims = [30, 25, 20, 12][:len(cons)]
    R = 4
    say("constraints", cons)
    X, _ = o.make_tensor(dims, R, seed=13, snr_db=30.0)
    init = o.gen_factors(dims, R, seed=14)
    h.set_tensor(X)
    kw = dict(max_iter=10, threshold_error=0.0, constraints=cons)
    for form, oform in ((P.MTTKRP_STANDARD, o.MTTKRP_STANDARD), (P.MTTKRP_DIMTREE, o.MTTKRP_DIMTREE)):
        Fg, stg, logg = _als_parity(h, X, R, init, mttkrp_form=form, oform=oform, **kw)
        for k, c in enumerate(cons):
            if c == 2:                                      # orthonormal columns
                assert np.allclose(Fg[k].T @ Fg[k], np.eye(R), atol=1e-10)
            if c == 4:                                      # constant: only rescaled (Normalize)
                ratio = Fg[k] / init[k]
                assert np.allclose(ratio, ratio[0:1, :], rtol=1e-12)


def test_work_buffers_shared_between_handles_and_threads():
    """Calls take their work buffers from a pool that the handles of a GPU share: calls of
    different sizes on four handles in four threads at once, with failing calls between them,
    give the bits that each handle gives alone."""
    import threading
    rng = np.random.default_rng(8)
    shapes = [((37, 23, 41), 5), ((120, 90, 70), 20), ((40, 31, 22, 9), 12), ((300, 64, 50), 40)]
    handles, calls = [], []
    for dims, R in shapes:
        hd = P.Handle(0)
        hd.set_tensor(rng.standard_normal(dims), storage=P.TENSOR_BOTH)
        A = [rng.random((I, R)) for I in dims]
        handles.append(hd)
        calls.append([lambda hd=hd, A=A: hd.mttkrp(A, 1), lambda hd=hd, A=A: hd.mttkrp_dimtree(A, arith=P.ARITH_F32),
                      lambda hd=hd, A=A, R=R: hd.cpd(R, A, max_iter=4, threshold_error=0.0)[0]])
    alone = [[c() for c in cs] for cs in calls]
    bad = []

    def work(k):
        for _ in range(5):
            try:
                handles[k].mttkrp([np.zeros((3, 65))], 0)     # rank above the limit
                bad.append(k)
            except P.PtnError:
                pass
            for c, want in zip(calls[k], alone[k]):
                got = c()
                same = all(np.array_equal(g, w) for g, w in zip(got, want)) if isinstance(want, list) else \
                    np.array_equal(got, want)
                if not same:
                    bad.append(k)
    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(shapes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for hd in handles:
        hd.close()
    assert not bad


def test_calls_that_fail_with_work_buffers_taken_leave_the_others_alone():
    """As above, with calls among them that run out of memory when they already hold work buffers: an
    NNLS solve whose iterates (256 x 2.6 million rows x 64 doubles, 341 GB) exceed the memory of the
    GPU after its row buffers were taken, which also empties the pool under the other threads.  Every
    worker reaches its end, every result has the bits of the call alone, and so have calls of the
    failing handle and of a new one afterwards."""
    import ctypes
    import threading
    rng = np.random.default_rng(9)
    shapes = [((37, 23, 41), 5), ((120, 90, 70), 20), ((40, 31, 22, 9), 12), ((300, 64, 50), 40)]
    square = np.eye(64)

    def out_of_memory(hd):
        # (the rows are not read before the iterates have their memory)
        it, L, mu = ctypes.c_int(), ctypes.c_double(), ctypes.c_double()
        p = square.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
        return P.lib().ptn_nesterov_mnls(hd._h, 2600000, 64, p, p, 1e-2, 1e-2, 255, p, ctypes.byref(it),
                                         ctypes.byref(L), ctypes.byref(mu))

    def calls_of(hd, dims, A, R):
        return [lambda: hd.mttkrp(A, 1), lambda: hd.mttkrp_dimtree(A, arith=P.ARITH_F32),
                lambda: hd.cpd(R, A, max_iter=4, threshold_error=0.0)[0]]

    def equal(got, want):
        return all(np.array_equal(g, w) for g, w in zip(got, want)) if isinstance(want, list) else \
            np.array_equal(got, want)

    tensors = [rng.standard_normal(dims) for dims, _ in shapes]
    starts = [[rng.random((I, R)) for I in dims] for dims, R in shapes]
    handles, calls = [], []
    for (dims, R), X, A in zip(shapes, tensors, starts):
        hd = P.Handle(0)
        hd.set_tensor(X, storage=P.TENSOR_BOTH)
        handles.append(hd)
        calls.append(calls_of(hd, dims, A, R))
    alone = [[c() for c in cs] for cs in calls]
    say("failing call alone")
    assert out_of_memory(handles[0]) == 2
    bad, done = [], []

    def work(k):
        try:
            for i in range(4):
                if k == 0 and out_of_memory(handles[0]) != 2:
                    bad.append((k, i, "ran"))
                for j, (c, want) in enumerate(zip(calls[k], alone[k])):
                    if not equal(c(), want):
                        bad.append((k, i, j))
            done.append(k)
        except BaseException as e:                          # an exception in a thread fails no test by itself
            bad.append((k, repr(e)))

    say("four threads")
    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(shapes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad and sorted(done) == list(range(len(shapes))), (bad, done)
    assert out_of_memory(handles[0]) == 2
    for c, want in zip(calls[0], alone[0]):
        assert equal(c(), want)
    with P.Handle(0) as hd:
        hd.set_tensor(tensors[1], storage=P.TENSOR_BOTH)
        for c, want in zip(calls_of(hd, shapes[1][0], starts[1], shapes[1][1]), alone[1]):
            assert equal(c(), want)
    for hd in handles:
        hd.close()


@pytest.mark.parametrize("R", [3, 32, 33, 64])
@pytest.mark.parametrize("dims", [(1, 7, 9), (3, 300, 5), (31, 17, 33), (32, 64, 5), (33, 20, 30), (50, 257, 3),
                                  (97, 10, 11), (130, 9, 8)])
def test_fp32_fibre_contraction_at_unaligned_lengths(h, dims, R):
    """The FP32 and bf16x3 contractions over mode 0 read fibres in 32-element steps wherever they
    start.  Small integers make every product and sum exact in both (below 2^24, 16 bits of
    split products), so the MTTKRPs of modes 1 and 2 must equal numpy's; an infinity at the start
    of a fibre stays in the rows that contain it, though the fibre before is read past its end."""
    rng = np.random.default_rng(R)
    X = rng.integers(-8, 9, dims).astype(np.float64)
    A = [rng.integers(-4, 5, (I, R)).astype(np.float64) for I in dims]
    for fill in (None, np.inf):
        if fill is not None:
            X[0, 3, 2] = fill
            A[0][0], A[1][3], A[2][2] = 1.0, 1.0, 1.0
        h.set_tensor(X, storage=P.TENSOR_F32)
        T = np.tensordot(A[0], X, axes=(0, 0))                       # R x I1 x I2
        clean = {1: np.arange(dims[1]) != 3, 2: np.arange(dims[2]) != 2}
        for arith in (P.ARITH_F32, P.ARITH_BF16X3):
            for mode in (1, 2):
                keep = clean[mode] if fill is not None else slice(None)
                with np.errstate(invalid="ignore"):
                    want = np.einsum("rjk,kr->jr", T, A[2]) if mode == 1 else np.einsum("rjk,jr->kr", T, A[1])
                got = h.mttkrp(A, mode, arith=arith)
                assert np.array_equal(got[keep], want[keep])
                if fill is not None:
                    assert not np.isfinite(got[~keep]).any()


@pytest.mark.parametrize("R", [7, 40])
@pytest.mark.parametrize("dims", [(31, 127, 129), (32, 127, 129), (33, 128, 129), (64, 160, 250), (65, 200, 331),
                                  (97, 256, 257), (96, 300, 301), (63, 400, 501), (40, 447, 450)])
def test_fp32_fibre_contraction_at_the_block_shapes_edges(h, dims, R):
    """Fibre counts below and above 16384, 65536 and 200000, where the block goes from one tile of
    32 fibres to 2 .. 5 to the blocks of 256, fibres of one half, one and several 64-element
    tiles.  Small integers: exact, as above."""
    rng = np.random.default_rng(R)
    X = rng.integers(-8, 9, dims).astype(np.float64)
    A = [rng.integers(-4, 5, (I, R)).astype(np.float64) for I in dims]
    h.set_tensor(X, storage=P.TENSOR_F32)
    T = np.tensordot(A[0], X, axes=(0, 0))
    want = np.einsum("rjk,kr->jr", T, A[2])
    for arith in (P.ARITH_F32, P.ARITH_BF16X3):
        assert np.array_equal(h.mttkrp(A, 1, arith=arith), want)


@pytest.mark.parametrize("dims", [(100, 100, 100), (60, 127, 128), (40, 50, 61, 85)])
def test_fp32_products_with_splits_past_the_last_column(h, dims):
    """k chunks are rounded up to 16 columns, so the last of many splits can start past the end
    (100^3, mode 0: 39 splits of 272 of 10000 columns); they add zero.  The tensor's memory is
    followed by that of a larger one, so a read past its end is not a read of zeros.  FP32 sums
    in splits of at most 272 products of order 1: 1e-5 relative."""
    rng = np.random.default_rng(5)
    h.set_tensor(rng.standard_normal((160, 160, 160)), storage=P.TENSOR_F32)
    X = rng.standard_normal(dims)
    A = [rng.standard_normal((I, 10)) for I in dims]
    h.set_tensor(X, storage=P.TENSOR_F32)
    want = X.reshape(dims[0], -1, order="F") @ np.array(
        [np.prod(v, axis=0) for v in _rows_of_khatri_rao(A[1:])])
    got = h.mttkrp(A, 0, arith=P.ARITH_F32), h.mttkrp_dimtree(A, arith=P.ARITH_F32)[0]
    for M in got:
        assert P.rel_err(M, want) <= 1e-5


def _rows_of_khatri_rao(A):
    for i in np.ndindex(*[a.shape[0] for a in A[::-1]]):
        yield [a[j] for a, j in zip(A, i[::-1])]


@pytest.mark.parametrize("R", [5, 17, 33, 64])
@pytest.mark.parametrize("I0", [1, 3, 15, 16, 17, 31, 33, 50, 97])
def test_fibre_contraction_at_unaligned_lengths(h, I0, R):
    """X x_0 A_0 on the FP64 matrix cores reads each fibre in 16-element blocks wherever it starts:
    every residue class of the fibre length, more fibres than one block holds, each column
    tile count, FP64 and FP32 tensors (the values are FP32 numbers, so both are exact), against
    numpy in FP64.  Sums of up to 97 x 31 products of order 1: 1e-13 relative."""
    rng = np.random.default_rng(I0 + 100 * R)
    X = rng.standard_normal((I0, 9, 31)).astype(np.float32).astype(np.float64)
    A = [rng.standard_normal((I, R)) for I in X.shape]
    h.set_tensor(X, storage=P.TENSOR_BOTH)
    T = np.tensordot(A[0], X, axes=(0, 0))                       # R x I1 x I2
    want = {1: np.einsum("rjk,kr->jr", T, A[2]), 2: np.einsum("rjk,jr->kr", T, A[1])}
    for arith in (P.ARITH_F64, P.ARITH_F32_F64):
        for mode in (1, 2):
            assert P.rel_err(h.mttkrp(A, mode, arith=arith), want[mode]) <= 1e-13


@pytest.mark.parametrize("R", [16, 33, 64])
@pytest.mark.parametrize("dims", [(19, 127, 129), (16, 129, 128), (35, 131, 127), (16, 256, 256), (21, 257, 257)])
def test_fibre_contraction_at_the_tile_counts_edges(h, dims, R):
    """The same contraction with just below and above 16384 and 65536 fibres, where a wave's share
    goes from 1 to 2 to 4 tiles of 16 fibres, whole and ragged.  Sums of up to 35 x 257 products
    of order 1: 1e-13 relative."""
    rng = np.random.default_rng(R)
    X = rng.standard_normal(dims).astype(np.float32).astype(np.float64)
    A = [rng.standard_normal((I, R)) for I in dims]
    h.set_tensor(X, storage=P.TENSOR_BOTH)
    T = np.tensordot(A[0], X, axes=(0, 0))
    want = np.einsum("rjk,kr->jr", T, A[2])
    for arith in (P.ARITH_F64, P.ARITH_F32_F64):
        assert P.rel_err(h.mttkrp(A, 1, arith=arith), want) <= 1e-13


@pytest.mark.parametrize("R", [1, 2, 3, 15, 16, 17, 32, 33, 63, 64])
def test_orthogonal_update_is_the_polar_factor_at_every_padded_rank(h, R):
    """One update of mode 0 under the orthogonality constraint, A = M (M^T M)^-1/2, against the
    SVD's polar factor of the same MTTKRP: even and odd ranks at the edges of the padded sizes.
    The condition of this M^T M is at most 510 (R = 64), so some hundred roundings of 1.1e-16
    leave the factor within 1e-11."""
    rng = np.random.default_rng(R)
    dims = [200, 9, 11]
    X, init = rng.standard_normal(dims), [rng.standard_normal((I, R)) for I in dims]
    h.set_tensor(X)
    F, _, _ = h.cpd(R, init, max_iter=1, threshold_error=0.0, normalization=0, constraints=[2, 4, 4])
    U, _, Wt = np.linalg.svd(h.mttkrp(init, 0), full_matrices=False)
    say("rank", R, np.abs(F[0] - U @ Wt).max())
    assert np.abs(F[0] - U @ Wt).max() <= 1e-11
    assert np.abs(F[0].T @ F[0] - np.eye(R)).max() <= 1e-11


@pytest.mark.parametrize("R", [2, 5, 16, 17, 33, 64])
@pytest.mark.parametrize("scale", [0, 230, -230, "graded", "zero column"])
def test_orthogonal_update_outside_the_short_operations_range(h, R, scale):
    """The rotations' divisions and roots take short forms while their operands lie within 2^+-400, and the
    operators elsewhere: tensors scaled by 2^+-230 (diagonals of M^T M about 2^+-460), columns of M from
    2^-110 to 2^110 of the others (rotation angles beyond 2^199) and a column of zeros.  Small integers times
    powers of two make M and its scalings exact in any order of sums, and everything after M is the
    oracle's operation by operation, so the factors agree bit for bit (NaN of a zero column included)."""
    rng = np.random.default_rng(R)
    dims = [70, 9, 11]
    X = rng.integers(-4, 5, dims).astype(np.float64)
    init = [rng.integers(-3, 4, (I, R)).astype(np.float64) for I in dims]
    if scale == "graded":
        init[1] *= 2.0 ** rng.integers(-110, 111, R)
    elif scale == "zero column":
        init[1][:, R // 2] = 0.0
    else:
        X *= 2.0 ** scale
    h.set_tensor(X)
    assert np.array_equal(h.mttkrp(init, 0), o.mttkrp(X, init, 0))
    kw = dict(max_iter=1, threshold_error=0.0, normalization=0, acceleration=0, constraints=[2, 4, 4])
    F, _, _ = h.cpd(R, init, **kw)
    Fo, _, _ = o.cpd(X, R, init, cost_form=o.COST_GRAM, **kw)
    say("rank", R, scale, "finite", np.isfinite(F[0]).all())
    assert np.array_equal(F[0], Fo[0], equal_nan=True)
    if scale not in ("zero column", "graded"):
        assert np.abs(F[0].T @ F[0] - np.eye(R)).max() <= 1e-9


@pytest.mark.parametrize("dims,R", [([6, 5, 7, 4, 5], 3), ([4, 5, 3, 4, 3, 4], 3), ([3, 4, 3, 2, 3, 2, 3], 2),
                                    ([3, 2, 3, 2, 2, 3, 2, 3], 2)])
def test_dimtree_higher_orders(h, dims, R):
    """Orders 5-8 in the tree: the root's children (modes [0, ceil(N/2)) and the rest), each
    one pass over X; every MTTKRP against the oracle's, FP64 and FP32 stream; the fused
    line-search pass against the unfused one; then ALS in the tree form against the
    oracle's standard form."""
    say("tree order", len(dims), dims)
    rng = np.random.default_rng(len(dims))
    X = np.asfortranarray(rng.standard_normal(dims))
    A = [rng.random((I, R)) for I in dims]
    h.set_tensor(X, storage=P.TENSOR_BOTH)
    D = h.mttkrp_dimtree(A)
    D32 = h.mttkrp_dimtree(A, arith=P.ARITH_F32_F64)
    for mode in range(len(dims)):
        ref = o.mttkrp(X, A, mode)
        assert P.rel_err(D[mode], ref) < 1e-13, mode
        assert P.rel_err(D32[mode], ref) < 1e-6, mode
    Xc, _ = o.make_tensor(dims, R, seed=len(dims) + 20, snr_db=30.0)
    init = o.gen_factors(dims, R, seed=len(dims) + 21)
    h.set_tensor(Xc, storage=P.TENSOR_BOTH)
    kw = dict(max_iter=8, threshold_error=0.0)
    _fused_equals_unfused(h, R, init, kw)
    _als_parity(h, Xc, R, init, mttkrp_form=P.MTTKRP_DIMTREE, **kw)


@pytest.mark.parametrize("dims", [[6, 7, 8], [70, 37, 45]])
def test_zero_column_fallback_on_gpu(h, dims):
    """A negative tensor drives every Nesterov solve to zero: each mode takes the
    0.9 A + 0.1 A_old fallback, and its Gram (one or several 32-row chunks) feeds the
    next modes, so every factor and the cost check the fallback's Gram too."""
    say("zero-column fallback", dims)
    rng = np.random.default_rng(12)
    X = -o.cp_full([rng.random((I, 2)) for I in dims])
    init = [rng.random((I, 3)) for I in dims]
    h.set_tensor(X)
    kw = dict(max_iter=2, threshold_error=0.0, normalization=0, acceleration=0)
    Fg, stg, logg = h.cpd(3, init, **kw)
    Fo, sto, logo = o.cpd(X, 3, init, cost_form=o.COST_GRAM, **kw)
    assert logg[0]["zero_col_fallback"][0] == 1
    assert [l["zero_col_fallback"] for l in logg] == [l["zero_col_fallback"] for l in logo]
    for a, b in zip(Fg, Fo):
        assert np.array_equal(a, b)
    assert stg["f_value"] == pytest.approx(sto["f_value"], rel=1e-12)


@pytest.mark.parametrize("R", [3, 17, 33, 49])
@pytest.mark.parametrize("dims", [[1, 31, 32], [33, 128, 129], [255, 256, 257], [300, 5, 4]])
def test_update_finish_at_the_row_chunks_edges(h, dims, R):
    """The end of an update (the stopping iterate, the zero-column test, the Gram) for row counts
    about the 32-row chunks and the eight partial sums added at a time, at every padded rank; a
    tensor with its sign turned takes the zero-column mix, upright it does where the oracle does.
    Against the oracle: the MTTKRPs
    agree to rounding, the rest operation by operation, so the factors within 1e-10."""
    rng = np.random.default_rng(R)
    A = [rng.random((I, 2)) for I in dims]
    init = [rng.random((I, R)) for I in dims]
    kw = dict(max_iter=2, threshold_error=0.0, normalization=0, acceleration=0)
    for sign in (1.0, -1.0):
        X = sign * o.cp_full(A)
        h.set_tensor(X)
        Fg, _, logg = h.cpd(R, init, **kw)
        Fo, _, logo = o.cpd(X, R, init, cost_form=o.COST_GRAM, **kw)
        assert [l["zero_col_fallback"] for l in logg] == [l["zero_col_fallback"] for l in logo]
        assert [l["nnls_iters"] for l in logg] == [l["nnls_iters"] for l in logo]
        assert sign > 0 or logg[0]["zero_col_fallback"][0] == 1
        for a, b in zip(Fg, Fo):
            assert P.rel_err(a, b) <= 1e-10


def test_invalid_arguments_raise(h):
    say("error paths")
    h.set_tensor(np.ones((4, 5, 6), order="F"))
    init = [np.ones((I, 3)) for I in (4, 5, 6)]
    with pytest.raises(P.PtnError):
        h.cpd(65, [np.ones((I, 65)) for I in (4, 5, 6)])          # rank above the wave-per-row limit
    with pytest.raises(P.PtnError):
        h.cpd(3, init, constraints=[1, 7, 1])                       # no such constraint
    with pytest.raises(P.PtnError):
        h.mttkrp(init, 5)                                           # bad mode
    with pytest.raises(P.PtnError):
        h.mttkrp(init, 0, arith=P.ARITH_F32_F64)                    # no FP32 copy uploaded
    h.set_tensor(np.ones((4, 5, 6), order="F"), storage=P.TENSOR_BOTH)
    with pytest.raises(P.PtnError):
        h.cpd(3, init, fuse_accel=1, arith=P.ARITH_F32)             # paired pass needs the tree
    with pytest.raises(P.PtnError):
        h.cpd(3, init, fuse_accel=1, mttkrp_form=P.MTTKRP_DIMTREE)  # ... and FP32-output contractions
