"""Parity of the HIP engine with the oracle (same seeded inputs, sizes the oracle finishes in
seconds) and, at the L=32, Nt=128 size, with closed forms.  Tolerances: FP64 path 1e-10
relative (log-det, force, M_hat), FP32-mixed force 1e-5 relative."""
import ctypes as C

import numpy as np
import pytest

import _dense as D
from _gpu import ephmc, gpu_context, rel, say
from _oracle import MT, OracleModel, oracle, ptr

pytestmark = pytest.mark.gpu


def field(om, seed, scale=1.0):
    return np.random.default_rng(seed).standard_normal(om.dim) * scale


@pytest.mark.parametrize("l1,l2,nt", [(1, 1, 4), (2, 2, 4), (2, 3, 8), (5, 4, 8), (6, 6, 32), (8, 12, 16), (16, 16, 8)])
def test_M_hat(l1, l2, nt):
    say("M_hat", l1, l2, nt)
    om = OracleModel(l1, l2, nt, beta=nt * 40 / 32)
    om.set_couplings(kappa=om.kappa * 10)
    ctx = gpu_context(om)
    np.testing.assert_array_equal(ctx.lattice(), om.nnt)
    x = field(om, nt)
    Mg = ctx.M_hat(x)
    Mo = om.M_hat(x)
    assert rel(Mg, Mo) < 1e-13


@pytest.mark.parametrize("n", [2, 33, 37, 63, 97, 1023])
def test_gj_trailing_blocks(n):
    """Block steps whose diagonal block is cut short (1, 5, 31, 1 and 31 columns; odd sizes pair
    the last pivot with an identity row): log det and inverse against numpy on the fast path."""
    say("gj trailing block", n)
    om = OracleModel(n, 1, 1)
    ctx = gpu_context(om)
    A = np.random.default_rng(n).standard_normal((n, n)) * 0.3 / np.sqrt(n) + np.eye(n) * 2
    A[0, 0] = -2                               # one negative pivot: sign -1
    ld, sg, inv = ctx.logdet_inv(A.T.copy().ravel())
    s0, l0 = np.linalg.slogdet(A)
    assert ld == pytest.approx(l0, rel=1e-12) and sg == int(s0) == -1
    assert rel(inv.reshape(n, n).T, np.linalg.inv(A)) < 1e-12
    assert ctx.gj_fallbacks() == 0


@pytest.mark.parametrize("strip", ["2", "4"])
@pytest.mark.parametrize("l1,l2,nt", [(2, 3, 4), (6, 6, 8), (16, 16, 8), (32, 32, 4)])
def test_strip_chain_bit_identical(monkeypatch, l1, l2, nt, strip):
    """The strip form of the slice stencil sums in the same order as the site-per-thread form:
    M_hat must agree to the last bit (EPHMC_CHAIN_STRIP=0 selects the site-per-thread form)."""
    say("strip vs site chain", l1, l2, nt, strip)
    om = OracleModel(l1, l2, nt, beta=nt * 40 / 32)
    ctx = gpu_context(om)
    x = field(om, 5)
    monkeypatch.setenv("EPHMC_CHAIN_STRIP", strip)
    Ms = ctx.M_hat(x)
    monkeypatch.setenv("EPHMC_CHAIN_STRIP", "0")
    Mg = ctx.M_hat(x)
    np.testing.assert_array_equal(Ms, Mg)


# every shape of the patch form (one site up to 512 / 640 sites, 2 x 2 sites beyond, more than 512
# threads), extents that are no multiple of the patch, lattices of one row or column, orders 2 and 6
@pytest.mark.parametrize("l1,l2,nt,order", [(1, 1, 2, 4), (5, 4, 3, 4), (1, 40, 3, 4), (64, 1, 3, 2), (16, 16, 3, 6), (21, 19, 3, 4),
                                            (25, 25, 3, 4), (27, 31, 3, 4), (32, 32, 3, 6), (33, 32, 2, 4), (700, 1, 2, 4),
                                            (1, 1001, 2, 4), (45, 45, 2, 4), (64, 32, 2, 2)])
def test_patch_chain_bit_identical(monkeypatch, l1, l2, nt, order):
    """The patch form of the chain sums in the order of the site form: M_hat (fp64) and the mixed
    molecular-dynamics force (fp32 chain) agree to the last bit (EPHMC_CHAIN_STRIP=0: the site form)."""
    say("patch vs site chain", l1, l2, nt, order)
    om = OracleModel(l1, l2, nt, beta=nt * 40 / 32, taylor=order)
    ctx = gpu_context(om, precision=1, taylor_order=order)
    x = field(om, 5)
    Mp, Fp = ctx.M_hat(x), ctx.md_force(x)
    monkeypatch.setenv("EPHMC_CHAIN_STRIP", "0")
    np.testing.assert_array_equal(Mp, ctx.M_hat(x))
    np.testing.assert_array_equal(Fp, ctx.md_force(x))


@pytest.mark.parametrize("revert,stop", [(0, 2), (0, 1), (0, 0), (1, 0), (1, -1)])
def test_apply_exp_partial(revert, stop):
    say("apply_exp_M", revert, stop)
    om = OracleModel(5, 4, 2)
    om.set_couplings(kappa=om.kappa * 10)
    ctx = gpu_context(om)
    x = field(om, 3)
    n = om.ns
    M = np.random.default_rng(1).standard_normal(n * n)
    g = ctx.apply_exp_M(x[:3 * n], M, revert, stop)
    o = M.copy()
    w = np.zeros(2 * n * n)
    oracle().orc_apply_exp_mu_K_to_M(om.ref, ptr(x), ptr(o), ptr(w), revert, stop)
    assert rel(g, o) < 1e-14


@pytest.mark.parametrize("n", [1, 5, 36, 100, 256, 300, 1024])
def test_logdet_inverse_random(n):
    say("gj random", n)
    om = OracleModel(n, 1, 1)
    ctx = gpu_context(om)
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n)) + np.eye(n) * (0 if n < 50 else 3)
    ld, sg, inv = ctx.logdet_inv(A.T.copy().ravel())
    s0, l0 = np.linalg.slogdet(A)
    assert ld == pytest.approx(l0, rel=1e-11, abs=1e-11) and sg == int(s0)
    assert rel(inv.reshape(n, n).T, np.linalg.inv(A)) < 1e-10
    # row exchanges are needed for these matrices exactly when LU without exchanges has a
    # multiplier above 1; then the pivoted fallback must have run
    import scipy.linalg as sl
    lu, piv = sl.lu_factor(A)
    needs = bool(np.any(piv != np.arange(n)))
    say("gj random", n, "row exchanges", needs, "fallbacks", ctx.gj_fallbacks())
    assert (ctx.gj_fallbacks() > 0) == needs


@pytest.mark.parametrize("n,r,j", [(256, 100, 97), (256, 200, 97), (1024, 610, 608), (1024, 900, 608)])
def test_gj_single_exchange_in_a_middle_block(n, r, j):
    """A diagonally dominant matrix with one entry |A[r][j]| > |A[j][j]| below the diagonal in the
    pivot column j of a block that is neither the first nor the last: LU needs one row exchange
    there (its multiplier is about 1.5), inside the diagonal block (r in the block of j) or below
    it.  The check must raise the flag, the pivoted fallback must run, and log det, sign and
    inverse equal numpy's."""
    say("gj exchange in a middle block", n, r, j)
    om = OracleModel(n, 1, 1)
    ctx = gpu_context(om)
    A = np.random.default_rng(n + r).standard_normal((n, n)) * 0.01 / np.sqrt(n) + np.eye(n) * 2
    A[r, j] = 3.0
    ld, sg, inv = ctx.logdet_inv(A.T.copy().ravel())
    s0, l0 = np.linalg.slogdet(A)
    assert ctx.gj_fallbacks() == 1
    assert ld == pytest.approx(l0, rel=1e-12) and sg == int(s0)
    assert rel(inv.reshape(n, n).T, np.linalg.inv(A)) < 1e-12
    A[r, j] = 1.5                              # multiplier 0.75: no exchange, fast path
    ld, sg, inv = ctx.logdet_inv(A.T.copy().ravel())
    assert ctx.gj_fallbacks() == 1
    assert ld == pytest.approx(np.linalg.slogdet(A)[1], rel=1e-12)


def test_logdet_inverse_diagonally_dominant_no_fallback():
    """A matrix whose multipliers are all below 1 (no exchanges) stays on the fast path."""
    n = 300
    om = OracleModel(n, 1, 1)
    ctx = gpu_context(om)
    A = np.random.default_rng(5).standard_normal((n, n)) * 0.01 + np.eye(n) * 2
    ld, sg, inv = ctx.logdet_inv(A.T.copy().ravel())
    s0, l0 = np.linalg.slogdet(A)
    assert ld == pytest.approx(l0, rel=1e-12) and sg == int(s0)
    assert rel(inv.reshape(n, n).T, np.linalg.inv(A)) < 1e-12
    assert ctx.gj_fallbacks() == 0


@pytest.mark.parametrize("n", [1, 3, 4, 15, 17, 31, 33, 47, 52, 63, 64, 65, 67, 95, 96, 97, 129, 160, 191, 1023, 1400, 1401, 1409, 1472, 1531])
def test_logdet_inverse_sizes(n):
    """Every form of the inversion at the edges of its range (one workgroup to N = 64, blocks of 32
    columns, blocks of 64 above N = 1400) and at last blocks of every kind: diagonally dominant with
    pivots of both signs, so that the fast path serves it, and the same matrix with one entry that
    asks for a row exchange late in it, so that the pivoted one does.  The condition numbers are of
    order 10 and numpy's own inverse is the reference: 1e-12 covers n eps kappa of both."""
    ctx = gpu_context(OracleModel(n, 1, 1))
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n)) * (0.3 / np.sqrt(n)) + np.diag(np.where(rng.random(n) < 0.3, -2.0, 2.0))
    for exchange in (False, True):
        if exchange:
            if n == 1:
                break
            A[n - 1, n - 2] = 6.0
        say("gj sizes", n, exchange)
        ld, sg, inv = ctx.logdet_inv(A.T.copy().ravel())
        s0, l0 = np.linalg.slogdet(A)
        assert ctx.gj_fallbacks() == int(exchange)
        assert ld == pytest.approx(l0, rel=1e-12) and sg == int(s0)
        assert rel(inv.reshape(n, n).T, np.linalg.inv(A)) < 1e-12


@pytest.mark.parametrize("l1,l2,nt", [(6, 6, 32), (16, 16, 64)])
def test_logdet_inverse_M_hat(l1, l2, nt):
    say("gj M_hat", l1, l2, nt)
    om = OracleModel(l1, l2, nt)
    ctx = gpu_context(om)
    x = field(om, 5)
    M = om.M_hat(x)
    ldo, so, invo = om.logdet_inv(M)
    ldg, sg, invg = ctx.logdet_inv(M)
    assert ldg == pytest.approx(ldo, rel=1e-12) and sg == so
    assert rel(invg, invo) < 1e-12
    assert ctx.gj_fallbacks() == 0


@pytest.mark.parametrize("l1,l2,nt,k", [(3, 3, 4, 16), (6, 6, 32, 16), (6, 6, 32, 5), (6, 6, 32, 1), (5, 7, 12, 4),
                                        (2, 2, 8, 3), (16, 16, 16, 8), (5, 7, 40, 1), (3, 3, 4, 1)])
def test_force_fp64(l1, l2, nt, k):
    say("force fp64", l1, l2, nt, k)
    om = OracleModel(l1, l2, nt, beta=nt * 40 / 32)
    om.set_couplings(kappa=om.kappa * 10)
    ctx = gpu_context(om, checkpoint=k)
    x = field(om, l1 + nt)
    ld, _, Minv = om.logdet_inv(om.M_hat(x))
    Fo = om.force(x, Minv, ld)
    Fg = ctx.force(x, Minv, ld)
    assert rel(Fg, Fo) < 1e-11


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("l1,l2,nt", [(6, 6, 40), (16, 16, 72), (32, 32, 8)])
def test_force_every_slice_matches_recompute(precision, l1, l2, nt):
    """k = 1 stores every partial product and the sweep reads them back (32 slices per launch);
    k = 8 recomputes them from checkpoints with the forward chain's arithmetic: same bits."""
    say("force k=1 vs k=8", precision, l1, l2, nt)
    om = OracleModel(l1, l2, nt, beta=nt * 40 / 32)
    x = field(om, 7)
    ref = gpu_context(om)
    _, _, Minv = ref.logdet_inv(ref.M_hat(x))
    F = {k: gpu_context(om, precision=precision, checkpoint=k).force(x, Minv, 0.0) for k in (1, 8)}
    np.testing.assert_array_equal(F[1], F[8])


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("l1,l2,nt", [(6, 6, 40), (32, 32, 8)])
def test_force_w0_order_bit_identical(monkeypatch, precision, l1, l2, nt):
    """The force sweep's two orders of the first W phase (its own barrier, or W_0 written at the
    end of the previous slice) do the same arithmetic in the same order: same bits."""
    say("force w0 order", precision, l1, l2, nt)
    om = OracleModel(l1, l2, nt, beta=nt * 40 / 32)
    x = field(om, 8)
    ref = gpu_context(om)
    _, _, Minv = ref.logdet_inv(ref.M_hat(x))
    F = {}
    for early in ("0", "1"):
        monkeypatch.setenv("EPHMC_ADJOINT_W0EARLY", early)
        F[early] = gpu_context(om, precision=precision, checkpoint=1).force(x, Minv, 0.0)
    np.testing.assert_array_equal(F["0"], F["1"])


@pytest.mark.parametrize("l1,l2", [(33, 32), (43, 43)])
def test_force_fp64_default_width_near_lds_limit(l1, l2):
    """FP64 force with the default column width at N = 1056 and 1849, the sizes where the sweep's
    reduction scratch decides whether C = 4 (or 2) still fits the 160 KiB of LDS: the default must
    pick a width that launches, and the force equals the oracle's."""
    say("force FP64 default width", l1, l2)
    om = OracleModel(l1, l2, 4, beta=4 * 40 / 32)
    ctx = gpu_context(om, checkpoint=1)
    x = field(om, 21)
    ld, _, Minv = ctx.logdet_inv(ctx.M_hat(x))
    Fg = ctx.force(x, Minv, ld)
    Fo = om.force(x, Minv, ld)
    say("rel err", rel(Fg, Fo))
    assert rel(Fg, Fo) < 1e-10


def test_maximum_lattice_size():
    """The largest lattice a context accepts, 64 x 32 = 2048 sites (Nt = 8; the chain and the sweep
    give each thread two sites): M_hat against the oracle (1e-13), log det and inverse against numpy
    (1e-10), and the force against the oracle's with the same inverse, FP64 (1e-10) with every slice
    stored and recomputed from checkpoints every 4 slices, mixed precision (1e-5).  One lattice row
    more (65 x 32 = 2080 sites) is refused as unsupported."""
    say("maximum lattice 64 x 32")
    om = OracleModel(64, 32, 8, beta=8 * 40 / 32)
    x = field(om, 31)
    n = om.ns
    Mo = om.M_hat(x)
    ctx = gpu_context(om, checkpoint=1)
    Mg = ctx.M_hat(x)
    say("M_hat rel err", rel(Mg, Mo))
    assert rel(Mg, Mo) < 1e-13
    ld, sg, Minv = ctx.logdet_inv(Mg)
    A, Ai = Mg.reshape(n, n).T, Minv.reshape(n, n).T
    sg_np, ld_np = np.linalg.slogdet(A)
    say("log det", ld, ld_np, "residual", np.abs(A @ Ai - np.eye(n)).max())
    assert sg == sg_np and abs(ld - ld_np) <= 1e-10 * max(1.0, abs(ld_np))
    assert np.abs(A @ Ai - np.eye(n)).max() < 1e-10
    Fo = om.force(x, Minv, ld)
    for prec, k, tol in ((0, 1, 1e-10), (0, 4, 1e-10), (1, 1, 1e-5)):
        c = ctx if (prec, k) == (0, 1) else gpu_context(om, precision=prec, checkpoint=k)
        Fg = c.force(x, Minv, ld)
        say("force precision %d checkpoint %d rel err %.2e" % (prec, k, rel(Fg, Fo)))
        assert rel(Fg, Fo) < tol
        if c is not ctx:
            c.close()
    ctx.close()
    with pytest.raises(ephmc().EphmcError, match="error -3"):
        gpu_context(OracleModel(65, 32, 8, beta=8 * 40 / 32))


def test_force_mixed():
    say("force mixed 6x6x32")
    om = OracleModel(6, 6, 32)
    ctx = gpu_context(om, precision=1)
    x = field(om, 2)
    ld, _, Minv = om.logdet_inv(om.M_hat(x))
    Fo = om.force(x, Minv, ld)
    Fg = ctx.force(x, Minv, ld)
    say("mixed force rel err", rel(Fg, Fo))
    assert rel(Fg, Fo) < 1e-5


@pytest.mark.parametrize("precision,tol", [(0, 1e-10), (1, 1e-5)])
@pytest.mark.parametrize("taylor", [2, 6, 8])
def test_taylor_orders(taylor, precision, tol):
    """Slice exponentials of Taylor orders 2, 6 and 8 (polynomial degree 2, 6, 8: one force-sweep
    instance per degree): M_hat and the force against the oracle built with the same order."""
    say("taylor order", taylor, "precision", precision)
    om = OracleModel(7, 5, 16, beta=16 * 40 / 32, taylor=taylor)
    ctx = gpu_context(om, precision=precision, taylor_order=taylor)
    x = field(om, 11)
    Mo = om.M_hat(x)
    assert rel(ctx.M_hat(x), Mo) < 1e-13
    ld, _, Minv = om.logdet_inv(Mo)
    Fo = om.force(x, Minv, ld)
    Fg = ctx.force(x, Minv, ld)
    say("rel err", rel(Fg, Fo))
    assert rel(Fg, Fo) < tol


@pytest.mark.parametrize("checkpoint", [1, 4])
@pytest.mark.parametrize("precision,tol", [(0, 1e-10), (1, 1e-5)])
@pytest.mark.parametrize("cols", ["1", "2", "4"])
@pytest.mark.parametrize("l1,l2,nt", [(7, 5, 8), (13, 11, 4), (23, 23, 4)])
def test_force_ragged(monkeypatch, l1, l2, nt, cols, precision, tol, checkpoint):
    """Force where the last workgroup's columns run past N (N = 35, 143, 529 are odd) and most
    lanes of a workgroup lie past the last site (N = 35 on 256 threads, 529 on 1024). In FP32
    those lanes load and gather but store nothing, and the columns past N read column N-1 and
    must add only zeros to the bond sums. Every slice stored (k = 1) and recomputed from every
    4th slice. beta = 40 Nt / 32 (slice width 1.25, as in the other force tests): with beta = 40 at
    Nt = 4 the slices are 10 wide and the FP32 chain keeps only about 3 digits."""
    say("force ragged", l1, l2, nt, "cols", cols, "precision", precision, "checkpoint", checkpoint)
    monkeypatch.setenv("EPHMC_ADJOINT_COLS", cols)
    om = OracleModel(l1, l2, nt, beta=nt * 40 / 32)
    ctx = gpu_context(om, precision=precision, checkpoint=checkpoint)
    x = field(om, 7)
    ld, _, Minv = om.logdet_inv(om.M_hat(x))
    Fo = om.force(x, Minv, ld)
    Fg = ctx.force(x, Minv, ld)
    say("rel err", rel(Fg, Fo))
    assert rel(Fg, Fo) < tol


# every number of stages (odd: one single stage), the largest transforms that LDS holds, direct sums
@pytest.mark.parametrize("nt", [1, 2, 4, 8, 16, 32, 64, 128, 256, 512, 1024, 3, 95, 590])
def test_boson_transforms_vs_numpy(nt):
    """Free-boson draw, momentum refresh, kinetic energy and exact flow against numpy's transforms; the
    direct sums add nt terms, so their rounding is nt eps at most."""
    say("boson transforms, nt =", nt)
    om = OracleModel(3, 1, nt)
    ctx = gpu_context(om)
    rng = np.random.default_rng(nt)
    n1, n2 = rng.standard_normal((2, nt, 9))
    f2 = om.omega + (2 * np.sin(np.pi * np.arange(nt // 2 + 1) / nt)) ** 2 / om.omega

    def scaled(a, g):
        return np.fft.irfft(np.fft.rfft(a, axis=0) * g[:, None], n=nt, axis=0) if nt > 1 else a * g[0]

    tol = 1e-13 * max(1, nt / 64) * max(1.0, (f2.max() / f2.min()) ** 0.5 * 1e-2)
    x, p = scaled(n1, f2 ** -.5), scaled(n2, f2 ** .5)
    assert rel(ctx.sample_free_bosons(n1.ravel()), x.ravel()) < tol
    assert rel(ctx.sample_fourier_momenta(n2.ravel()), p.ravel()) < tol
    assert ctx.energy_momenta(p.ravel()) == pytest.approx(.5 * (n2 ** 2).sum(), rel=1e-11)
    gx, gp = ctx.evolve_bosons(x.ravel(), p.ravel(), 0.3)
    assert rel(gx, (np.cos(.3) * x + np.sin(.3) * scaled(p, 1 / f2)).ravel()) < 10 * tol
    assert rel(gp, (np.cos(.3) * p - np.sin(.3) * scaled(x, f2)).ravel()) < 10 * tol


@pytest.mark.parametrize("nt", [1, 2, 8, 12, 32, 48])
def test_boson_kernels(nt):
    say("bosons", nt)
    om = OracleModel(3, 2, nt)
    ctx = gpu_context(om)
    lib = oracle()
    rng = np.random.default_rng(nt)
    x = rng.standard_normal(om.dim)
    p = rng.standard_normal(om.dim)
    xg, pg = ctx.evolve_bosons(x, p, 0.41)
    xo, po = x.copy(), p.copy()
    lib.orc_evolve_bosons(om.ref, ptr(xo), ptr(po), 0.41)
    assert rel(xg, xo) < 1e-13 and rel(pg, po) < 1e-13
    assert ctx.energy_momenta(p) == pytest.approx(lib.orc_energy_momenta(om.ref, ptr(p)), rel=1e-13)
    assert ctx.hamilton(x, 1.25, 3.5) == pytest.approx(lib.orc_hamilton(om.ref, ptr(x), 1.25, 3.5), rel=1e-13)
    for fn_g, fn_o in ((ctx.sample_fourier_momenta, lib.orc_sample_fourier_momenta),
                       (ctx.sample_free_bosons, lib.orc_sample_free_bosons)):
        st, st2 = MT(), MT()
        lib.orc_mt_seed(C.byref(st), 77)
        lib.orc_mt_seed(C.byref(st2), 77)
        normals = np.zeros(om.dim)
        lib.orc_random_vector(C.byref(st), ptr(normals), om.dim)
        out_o = np.zeros(om.dim)
        fn_o(om.ref, C.byref(st2), ptr(out_o))
        assert rel(fn_g(normals), out_o) < 1e-13


def test_hmc_accept_sequence_and_logdet():
    """Seeded FP64 chain at L=6, Nt=32, Nmd=10: identical accept/reject decisions and log-det
    within 1e-10 relative over the first 100 trajectories (oracle with the same RNG stream)."""
    om = OracleModel(6, 6, 32)
    lib = oracle()
    from _oracle import HMC
    h = HMC()
    assert lib.orc_hmc_init(C.byref(h), C.byref(om.m), 1, 10, 0.0, None) == 0
    ctx = gpu_context(om, steps=10)
    # same RNG stream: the chain's free-boson draw, then per trajectory dim normals + 1 uniform
    rng = MT()
    lib.orc_mt_seed(C.byref(rng), 1)
    normals = np.zeros(om.dim)
    lib.orc_random_vector(C.byref(rng), ptr(normals), om.dim)
    ctx.chain_init(normals)
    assert ctx.chain_logdet() == pytest.approx(h.logdet, rel=1e-12)
    dH = C.c_double()
    worst = 0.0
    for it in range(100):
        lib.orc_random_vector(C.byref(rng), ptr(normals), om.dim)
        u = lib.orc_mt_real2(C.byref(rng))
        acc_o = lib.orc_trajectory(C.byref(h), None, None, C.byref(dH), None, None)
        rec = ctx.trajectory(normals, u)
        worst = max(worst, abs(rec.logdet - h.logdet) / abs(h.logdet))
        assert rec.accepted == acc_o, "trajectory %d: gpu %d oracle %d (dH gpu %g oracle %g)" % (
            it, rec.accepted, acc_o, rec.dH, dH.value)
        assert abs(rec.dH - dH.value) < 1e-8
    say("100 trajectories, worst logdet rel diff", worst)
    assert worst < 1e-10
    lib.orc_hmc_free(C.byref(h))


# ---- full-size (L = 32, Nt = 128) properties -----------------------------------------------

def test_full_size_logdet_closed_form():
    say("closed-form logdet 32x32x128")
    om = OracleModel(32, 32, 128)
    ctx = gpu_context(om)
    u = np.random.default_rng(3).standard_normal((128, 3))
    x = D.uniform_field(32, 32, 128, u)
    ld, sg, _ = ctx.logdet_inv(ctx.M_hat(x))
    ref = D.closed_form_logdet(32, 32, 128, om.t, om.kappa, om.mu, u)
    say("logdet", ld, "closed form", ref)
    assert ld == pytest.approx(ref, rel=1e-10) and sg == 1


@pytest.mark.parametrize("precision,tol", [(0, 1e-10), (1, 1e-5)])
def test_full_size_force_closed_form(precision, tol):
    say("closed-form force 32x32x128 precision", precision)
    om = OracleModel(32, 32, 128)
    ctx = gpu_context(om, precision=precision, checkpoint=16)
    u = np.random.default_rng(4).standard_normal((128, 3)) * 2
    x = D.uniform_field(32, 32, 128, u)
    ld, _, minv = ctx.logdet_inv(ctx.M_hat(x))
    F = ctx.force(x, minv, ld)
    ref = D.closed_form_force(32, 32, 128, om.t, om.kappa, om.mu, u, om.flavors)
    say("force rel err", rel(F, ref))
    assert rel(F, ref) < tol


def test_full_size_force_finite_differences():
    """Adjoint force vs finite differences of the FP64 log det on 64 random components at 32x32,
    Nt = 128.  The log det carries about 1.5e-14 of rounding noise, so a central difference at eps
    has a noise of about 1.5e-14 / (2 eps) (relative 8e-6 at eps = 1e-5 for these forces of order
    1e-5), while its truncation O(eps^2) is far smaller here (the central difference at 4e-2 is
    within 1e-8).  Checked: central differences at eps = 1e-5, within 5e-5 (noise bound), and the
    Richardson extrapolation of the central differences at 2e-2 and 4e-2 (truncation O(eps^4)),
    within 1e-7 (measured 1.3e-8)."""
    om = OracleModel(32, 32, 128)
    ctx = gpu_context(om, checkpoint=16)
    x = field(om, 9)
    ld, _, minv = ctx.logdet_inv(ctx.M_hat(x))
    F = ctx.force(x, minv, ld)
    idx = np.random.default_rng(64).choice(om.dim, 64, replace=False)

    def central(i, eps):
        xp, xm = x.copy(), x.copy()
        xp[i] += eps
        xm[i] -= eps
        return om.flavors * (ctx.logdet_inv(ctx.M_hat(xp))[0] - ctx.logdet_inv(ctx.M_hat(xm))[0]) / (2 * eps)

    fd5 = np.array([central(i, 1e-5) for i in idx])
    err5 = rel(F[idx], fd5)
    fd = np.array([(4 * central(i, 2e-2) - central(i, 4e-2)) / 3 for i in idx])
    err = rel(F[idx], fd)
    say("finite-difference rel err: central eps 1e-5 %.2e, Richardson (2e-2, 4e-2) %.2e" % (err5, err))
    assert err5 < 5e-5
    assert err < 1e-7


@pytest.mark.parametrize("l1,l2,nt,order,prec", [(1, 1, 3, 4, 0), (2, 3, 1, 4, 0), (3, 5, 2, 2, 0), (16, 16, 5, 4, 0), (16, 16, 4, 6, 1),
                                                 (17, 16, 6, 4, 0), (21, 19, 7, 4, 0), (21, 19, 5, 2, 1), (23, 22, 3, 8, 0),
                                                 (24, 24, 4, 4, 1), (32, 32, 3, 4, 0), (33, 32, 3, 4, 0), (36, 36, 2, 6, 1)])
def test_force_sweep_columns(l1, l2, nt, order, prec, monkeypatch):
    """Odd and even numbers of slices, every polynomial degree and launch size: the force sweep gives the
    oracle's force at every number of columns per workgroup, and the same bits with W_0 written ahead
    or not and from a recomputed T.  1e-11 (fp64) and 1e-5 (fp32) as for every force here."""
    om = OracleModel(l1, l2, nt, beta=nt * 40 / 32, taylor=order)
    x = field(om, 9)
    monkeypatch.setenv("EPHMC_ADJOINT_COLS", "1")
    base = gpu_context(om, taylor_order=order)
    _, _, Minv = base.logdet_inv(base.M_hat(x))
    # (beyond the sizes that the oracle finishes in seconds: the fp64 sweep of one column per workgroup)
    ref = om.force(x, Minv, 0.0) if om.ns <= 400 else base.force(x, Minv, 0.0)
    tol = 1e-5 if prec else 1e-11
    for cols in (1, 2, 4):
        monkeypatch.setenv("EPHMC_ADJOINT_COLS", str(cols))
        bits = []
        for early, ckpt in (("0", 1), ("1", 1), ("1", 2)):
            monkeypatch.setenv("EPHMC_ADJOINT_W0EARLY", early)
            say("sweep", l1, l2, nt, order, prec, cols, early, ckpt)
            ctx = gpu_context(om, precision=prec, checkpoint=ckpt, taylor_order=order)
            try:
                bits.append(ctx.force(x, Minv, 0.0))
            except ephmc().EphmcError:
                assert l1 * l2 > 1024 and not prec and cols == 4     # over the LDS, as before
                continue
            assert rel(bits[-1], ref) < tol
            np.testing.assert_array_equal(bits[-1], bits[0])


def test_more_slices_than_a_grid_axis():
    """40000 slices: 80000 rows of coefficients, beyond the 65535 workgroups of a grid's second axis.
    M_hat, log det and force against the oracle; each slice rounds by about 10 eps at most, so 1e-10
    for the product and 1e-9 for the force, which multiplies two such products with the inverse."""
    om = OracleModel(3, 2, 40000)
    ctx = gpu_context(om, checkpoint=0)
    x = np.random.default_rng(4).standard_normal(om.dim)
    say("40000 slices")
    M = om.M_hat(x)
    assert rel(ctx.M_hat(x), M) < 1e-10
    ld, _, inv = om.logdet_inv(M)
    assert ctx.logdet_inv(M)[0] == pytest.approx(ld, rel=1e-10)
    assert rel(ctx.force(x, inv, ld), om.force(x, inv, ld)) < 1e-9


@pytest.mark.parametrize("l1,l2", [(24, 24), (32, 32)])
@pytest.mark.parametrize("taylor", [6, 8])
def test_force_sweep_width_of_high_orders(l1, l2, taylor, monkeypatch):
    """FP64 sweeps of Taylor orders 6 and 8 take two columns per workgroup between 513 and 1024 sites (four
    spill: 24x24 at order 8 690 against 456 us per 32 slices): the same bits as with two asked for, which
    group the partial sums unlike four."""
    om = OracleModel(l1, l2, 4, beta=5.0, taylor=taylor)
    x = np.random.default_rng(taylor).standard_normal(om.dim)
    say("sweep width", l1, l2, taylor)
    force = {}
    for cols in (None, "2", "4"):
        if cols:
            monkeypatch.setenv("EPHMC_ADJOINT_COLS", cols)
        force[cols] = gpu_context(om, checkpoint=0, taylor_order=taylor).md_force(x)
    np.testing.assert_array_equal(force[None], force["2"])
    assert not np.array_equal(force[None], force["4"])
