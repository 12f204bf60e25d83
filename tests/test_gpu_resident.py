"""Solves with the system held on the chip (glx_resident.h): CG on D^dag D in
the reference's order, single-pass and mixed precision, and the even/odd
solves, at the sizes where the tiling can go wrong -- strips of one column
count and of two, 60 and 61 columns, bands whose last one shares rows with the
band before it, every number of rows per wave, lattices of one tile, odd sizes
-- and the way back to a launch per iteration when a wait runs out.  Each test
also counts the solves that ran resident and those that gave up."""
import threading

import numpy as np
import pytest

from helpers import ENVELOPE, bicgstab_envelope, eo_envelope, lattice_inputs, relerr, resident_solves

pytestmark = pytest.mark.gpu

# lx, ly: 4 and 60 columns in one strip, 61 in two; ly = 8 one band, 9 a last
# band sharing 7 rows; 512 to 1020 rows take 3 to 10 rows per wave with the
# strips they have
SIZES = [(4, 8), (5, 9), (60, 8), (61, 23), (64, 16), (130, 70), (97, 301), (330, 222)]
LARGE = [(300, 512), (512, 400), (700, 512), (780, 780), (1000, 900)]


def system(glx, orc, lx, ly, beta=6.25):
    links, b, _ = lattice_inputs(orc, lx, ly, beta=beta, seed=1000 + lx + 3 * ly)
    return links, b, glx.Lattice(links, lx, ly), glx.DeviceArray(b)


@pytest.mark.parametrize("lx,ly", SIZES)
def test_cg_matches_oracle(glx, orc, lx, ly):
    """Reference order: the iterations and ops_count of the oracle with its
    serial or its correctly rounded sums (60 x 8: 125 and 124, 130 x 70: 178
    and 177), x to the bound the staggered solver tests use; single-pass:
    within 2 iterations."""
    m = 0.1
    links, b, lat, db = system(glx, orc, lx, ly)
    kw = dict(links=links, mass=m, lx=lx, ly=ly, max_iter=5000, eps=1e-10)
    runs = [orc.solve("cg", "staggered_normal", b, None, reductions=red, **kw) for red in ("serial", "extended")]
    dx = glx.DeviceArray(np.zeros_like(b))
    with resident_solves(glx, 1):
        ig = glx.dev_solve("cg", lat, "staggered_normal", m, dx, db, max_iter=5000)
    assert ig.iter in [io.iter for _, io in runs]
    xo, io = next(r for r in runs if r[1].iter == ig.iter)
    assert (ig.ops_count, ig.success) == (io.ops_count, io.success)
    assert relerr(dx.download(), xo) < 1e-11
    dx.upload(np.zeros_like(b))
    with resident_solves(glx, 1):
        jg = glx.dev_cg_fused(lat, "staggered_normal", m, dx, db, max_iter=5000)
    assert abs(jg.iter - io.iter) <= 2 and jg.success
    r = b - orc.apply("staggered_normal", dx.download(), links, m, lx, ly)
    # (A x is rounded to 4 u |x|, and |x| <= |b| / m^2 = 100 |b|: 1e-13 |b|)
    assert np.linalg.norm(r) <= 1.001e-10 * np.linalg.norm(b)
    assert abs(np.sqrt(jg.resSq) - np.linalg.norm(r)) <= 1e-13 * np.linalg.norm(b)


@pytest.mark.parametrize("links_prec", [1, 2])
@pytest.mark.parametrize("lx,ly", SIZES)
def test_mixed_matches_oracle(glx, orc, lx, ly, links_prec):
    m = 0.1
    links, b, lat, db = system(glx, orc, lx, ly)
    xs, _ = orc.solve("cg", "staggered_normal", b, None, links=links, mass=m, lx=lx, ly=ly, max_iter=5000, eps=1e-13)
    dx = glx.DeviceArray(np.zeros_like(b))
    with resident_solves(glx, 1):
        info = glx.dev_cg_mixed(lat, "staggered_normal", m, dx, db, link_prec=links_prec)
    x = dx.download()
    r = b - orc.apply("staggered_normal", x, links, m, lx, ly)
    assert info.success and info.reliable_updates > 0
    assert np.linalg.norm(r) <= 1.001e-10 * np.linalg.norm(b)
    # |x - x*| = |A^-1 r| <= |r| / m^2 (and x* is good to 1e-13 |b| / m^2)
    assert np.linalg.norm(x - xs) <= 1.01e-10 * np.linalg.norm(b) / m**2


@pytest.mark.parametrize("on", [True, False], ids=["resident", "launches"])
@pytest.mark.parametrize("lx,ly", [(61, 23), (330, 222), (780, 780)])
def test_mixed_adds_to_the_solution_in_fp64(glx, orc, resident, lx, ly, on):
    """A reliable update is x64 += x32 + alpha p in FP64 with alpha in FP64.
    After one iteration x32 = 0 and p = b, exact in FP32 here, so every
    entry of x / b is the one alpha to a few FP64 roundings (in FP32 they
    would differ by 1e-7); alpha itself is the FP64 one to the FP32 hops'
    rounding."""
    resident(on)
    m = 0.1
    links, b, _ = lattice_inputs(orc, lx, ly, beta=6.25, seed=1000 + lx + 3 * ly)
    b = b.astype(np.complex64).astype(np.complex128)
    dx = glx.DeviceArray(np.zeros_like(b))
    with resident_solves(glx, int(on)):
        info = glx.dev_cg_mixed(glx.Lattice(links, lx, ly), "staggered_normal", m, dx, glx.DeviceArray(b), max_iter=1)
    assert info.iter == 1 and info.reliable_updates == 1
    alpha = dx.download() / b
    want = np.vdot(b, b).real / np.vdot(b, orc.apply("staggered_normal", b, links, m, lx, ly)).real
    # (a complex product and quotient: 4 roundings each)
    assert np.max(np.abs(alpha - alpha[0])) <= 16 * np.finfo(float).eps * abs(alpha[0])
    assert abs(alpha[0] - want) <= 1e-6 * want


@pytest.mark.parametrize("lx,ly", LARGE)
def test_large_tiles_match_the_launch_per_iteration(glx, orc, resident, lx, ly):
    """Both run the same algorithm; their solutions stop at the same residual
    (1e-10 on a system of condition 1e3) within an iteration of each other."""
    m = 0.1
    links, b, lat, db = system(glx, orc, lx, ly)
    out = {}
    for on in (False, True):
        resident(on)
        for name in ("cg", "fused", "mixed"):
            dx = glx.DeviceArray(np.zeros_like(b))
            with resident_solves(glx, int(on)):
                if name == "cg":
                    info = glx.dev_solve("cg", lat, "staggered_normal", m, dx, db)
                elif name == "fused":
                    info = glx.dev_cg_fused(lat, "staggered_normal", m, dx, db)
                else:
                    info = glx.dev_cg_mixed(lat, "staggered_normal", m, dx, db)
            assert info.success
            out[name, on] = (info, dx.download())
    for name in ("cg", "fused", "mixed"):
        (i0, x0), (i1, x1) = out[name, False], out[name, True]
        assert abs(i0.iter - i1.iter) <= (1 if name != "mixed" else max(6, 0.03 * i0.iter)), name
        assert relerr(x1, x0) < 1e-10, name


@pytest.mark.parametrize("lx,ly", [(128, 8), (256, 72), (384, 100)])
@pytest.mark.parametrize("method", ["cg", "cg_fused", "mixed", "mixed_f16"])
def test_even_odd(glx, orc, lx, ly, method):
    m = 0.1
    links, b, lat, db = system(glx, orc, lx, ly)
    xs, err = eo_envelope(orc, b, links, m, lx, ly)
    dx = glx.DeviceArray(np.zeros_like(b))
    with resident_solves(glx, 1):
        info, _ = glx.dev_solve_staggered_eo(lat, m, dx, db, method)
    assert info.success
    assert relerr(dx.download(), xs) <= ENVELOPE * err


HOP_SIZES = [(2, 8), (7, 9), (62, 8), (63, 23), (64, 64), (130, 70), (97, 301), (300, 520)]


@pytest.mark.parametrize("op", ["laplace_real", "laplace", "laplace_u1"])
@pytest.mark.parametrize("lx,ly", HOP_SIZES)
def test_one_hop_cg_matches_oracle(glx, orc, lx, ly, op):
    """CG on the Laplacians through the host interface: the oracle's
    iterations (one apart where the last residual is within rounding of the
    tolerance), and |x - x*| <= |r| / m^2 with m^2 = 0.05 the gap."""
    links, bc, br = lattice_inputs(orc, lx, ly, beta=6.25, seed=500 + lx + ly)
    b = br if op == "laplace_real" else bc
    kw = dict(links=links, mass=0.05, lx=lx, ly=ly, max_iter=5000)
    xs, _ = orc.solve("cg", op, b, None, eps=1e-13, **kw)
    xo, io = orc.solve("cg", op, b, None, eps=1e-10, **kw)
    with resident_solves(glx, 1):
        xg, ig = glx.minv_vector_cg(op, b, eps=1e-10, **kw)
    assert ig.success and abs(ig.iter - io.iter) <= 1 and ig.ops_count == ig.iter + 2
    if ig.iter == io.iter:
        assert relerr(xg, xo) < 1e-11
    r = b - orc.apply(op, xg, links, 0.05, lx, ly)
    assert np.linalg.norm(r) <= 1.001e-10 * np.linalg.norm(b)
    assert np.linalg.norm(xg - xs) <= 1.01e-10 * np.linalg.norm(b) / 0.05


@pytest.mark.parametrize("op,mass", [("staggered", 0.2), ("staggered_dagger", 0.2), ("laplace_u1", 0.05), ("laplace", 0.05)])
@pytest.mark.parametrize("lx,ly", HOP_SIZES)
def test_one_hop_bicgstab(glx, orc, lx, ly, op, mass):
    """BiCGStab's path depends on rounding: iterations within the range of the
    oracle's on b and eight 1-ulp perturbations of it (97 x 301, laplace: 86 to
    97), widened by its own width on either side; the true residual as
    reported."""
    links, b, _ = lattice_inputs(orc, lx, ly, beta=6.25, seed=600 + lx + ly)
    kw = dict(links=links, mass=mass, lx=lx, ly=ly, max_iter=5000)
    with resident_solves(glx, 1):
        xg, ig = glx.minv_vector_bicgstab(op, b, eps=1e-10, **kw)
    _, _, its, _ = bicgstab_envelope(orc, op, b, dict(kw, eps=1e-10))
    width = max(2, its.max() - its.min())
    assert ig.success and ig.ops_count == 2 * ig.iter + 2
    assert its.min() - width <= ig.iter <= its.max() + width
    r = b - orc.apply(op, xg, links, mass, lx, ly)
    assert np.linalg.norm(r) <= 1e-9 * np.linalg.norm(b)
    assert abs(np.sqrt(ig.resSq) - np.linalg.norm(r)) <= 1e-12 * np.linalg.norm(b)


@pytest.mark.parametrize("solver", ["cg", "bicgstab"])
@pytest.mark.parametrize("op", ["laplace", "laplace_real", "laplace_u1"])
def test_laplacians_on_a_lattice_with_links(glx, orc, solver, op):
    """The free Laplacians take only their dimensions from a lattice, whose
    links are far from unit here; laplace_u1 takes both.  The residual is the
    oracle's operator's, as reported."""
    lx, ly, m = 61, 23, 0.05
    links, bc, br = lattice_inputs(orc, lx, ly, beta=2.0, seed=77)
    b = br if op == "laplace_real" else bc
    dx = glx.DeviceArray(np.zeros_like(b))
    # (BiCGStab on the real Laplacian has no resident kernel)
    with resident_solves(glx, 0 if (solver, op) == ("bicgstab", "laplace_real") else 1):
        info = glx.dev_solve(solver, glx.Lattice(links, lx, ly), op, m, dx, glx.DeviceArray(b), max_iter=5000, eps=1e-10)
    r = b - orc.apply(op, dx.download(), links, m, lx, ly)
    nb = np.linalg.norm(b)
    # (BiCGStab's iterated residual may drift from the true one)
    assert info.success and np.linalg.norm(r) <= (1e-9 if solver == "bicgstab" else 1.001e-10) * nb
    assert abs(np.sqrt(info.resSq) - np.linalg.norm(r)) <= 1e-12 * nb


@pytest.mark.parametrize("lx,ly,n_shift,freq", [(4, 8, 1, 1), (4, 8, 16, 10), (60, 9, 5, 3), (61, 23, 16, 10),
                                                (130, 70, 2, 7), (200, 144, 12, 10)])
def test_multishift_matches_oracle(glx, orc, runs_resident, lx, ly, n_shift, freq):
    """Every shift's solution and residual, and the iterations (a check apart
    where a shift crosses the tolerance within rounding)."""
    m = 0.1
    links, b, lat, db = system(glx, orc, lx, ly)
    shifts = 10.0 ** np.linspace(-3.0, 2.5, n_shift)
    kw = dict(links=links, mass=m, lx=lx, ly=ly, resid_freq_check=freq, max_iter=5000, eps=1e-10)
    X, io, _, _ = orc.cg_m("staggered_normal", b, shifts, **kw)
    xs = [glx.DeviceArray(b) for _ in shifts]  # (what they hold is overwritten)
    with resident_solves(glx, int(runs_resident)):
        ig = glx.dev_cg_m(lat, "staggered_normal", m, xs, db, shifts, resid_freq_check=freq, max_iter=5000)
    assert ig.success and abs(ig.iter - io.iter) <= freq and ig.ops_count == ig.iter + n_shift
    nb = np.linalg.norm(b)
    for k, s in enumerate(shifts):
        x = xs[k].download()
        r = b - orc.apply("staggered_normal", x, links, m, lx, ly) - s * x
        assert abs(np.sqrt(ig.resSqmrhs[k]) - np.linalg.norm(r)) <= 1e-12 * nb
        assert np.linalg.norm(r) <= 2e-10 * nb
        # both are within |r| / (m^2 + s) of the solution
        assert np.linalg.norm(x - X[k]) <= 4e-10 * nb / (m * m + s)


def test_multishift_stops_at_max_iter(glx, orc):
    lx, ly, m = 61, 23, 0.1
    links, b, lat, db = system(glx, orc, lx, ly)
    shifts = [0.0, 0.01, 1.0]
    for stop in (1, 2, 11):
        X, io, _, _ = orc.cg_m("staggered_normal", b, shifts, links=links, mass=m, lx=lx, ly=ly, resid_freq_check=10,
                               max_iter=stop, eps=1e-10)
        xs = [glx.DeviceArray(np.zeros_like(b)) for _ in shifts]
        with resident_solves(glx, 1):
            ig = glx.dev_cg_m(lat, "staggered_normal", m, xs, db, shifts, max_iter=stop)
        assert (ig.iter, ig.success, ig.ops_count) == (io.iter, io.success, io.ops_count)
        for x, xo in zip(xs, X):
            assert relerr(x.download(), xo) < 1e-12


# lx, ly, nc, two: one site and one block; wraps onto itself; last blocks with
# few sites; a site of 12 colours in 64 entries; two and four entries per lane;
# more colours than lanes
STENCILS = [(1, 1, 1, False), (6, 5, 1, False), (3, 2, 12, True), (16, 12, 4, True), (33, 31, 3, True),
            (32, 32, 8, False), (48, 48, 12, True), (64, 70, 12, False), (40, 40, 24, False), (7, 5, 70, False)]


def coarse(glx, orc, lx, ly, nc, two):
    """Identity plus random terms of spectral radius 1/2, all shifts on."""
    rng = np.random.default_rng(lx + 7 * ly + 31 * nc)
    o = orc.CStencil.random(rng, lx, ly, nc, two, shifts=(0.1 + 0.05j, -0.05j, 0.1))
    scale = 0.5 / np.sqrt(2.0 * nc * (13 if two else 5))
    o.hopping *= scale
    if two:
        o.two_link *= scale
    o.clover = (scale * o.clover.reshape(-1, nc, nc) + np.eye(nc)).reshape(-1)
    g = glx.StencilNc(lx, ly, nc, o.clover, o.hopping, o.two_link if two else None, o.shift, o.eo_shift, o.dof_shift, 0)
    b, x0 = (rng.standard_normal(o.n) + 1j * rng.standard_normal(o.n) for _ in range(2))
    return o, glx.CStencilDev(g), b, x0


def gcr_both(glx, resident, h, b, x0, **kw):
    """(x, info) on the chip and with a launch per phase."""
    out = []
    for on in (True, False):
        resident(on, 0)
        dx = glx.DeviceArray(x0)
        with resident_solves(glx, int(on)):
            info = h.solve("gcr", dx, glx.DeviceArray(b), **kw)
        out.append((dx.download(), info))
    return out


@pytest.mark.parametrize("lx,ly,nc,two", STENCILS)
def test_gcr_on_the_general_stencil(glx, orc, resident, lx, ly, nc, two):
    """The iterations of the launch-per-phase form (one apart where the norm
    meets the tolerance within rounding) and its iterates; the residual by the
    oracle's operator."""
    print(f"case {lx} x {ly} nc={nc} two={two}", flush=True)
    o, h, b, x0 = coarse(glx, orc, lx, ly, nc, two)
    nb = np.linalg.norm(b)
    (x, i), (xl, il) = gcr_both(glx, resident, h, b, x0, max_iter=400, eps=1e-10)
    assert i.success and il.success and abs(i.iter - il.iter) <= 1 and i.ops_count == i.iter + 2
    r = b - orc.cstencil_apply(o, x)
    assert np.linalg.norm(r) <= 1.01e-10 * nb
    # (entries of A x are sums of 13 nc products at most)
    assert abs(np.sqrt(i.resSq) - np.linalg.norm(r)) <= 13 * nc * 1e-15 * nb
    if lx * ly * nc > 60:  # (a small system is solved within so few)
        for stop in (1, 2, 7):
            (x, i), (xl, il) = gcr_both(glx, resident, h, b, x0, max_iter=stop, eps=1e-10)
            assert (i.iter, i.success, i.ops_count) == (il.iter, il.success, il.ops_count)
            assert relerr(x, xl) < 1e-12 and abs(i.resSq - il.resSq) <= 1e-10 * il.resSq


def test_gcr_over_several_launches(glx, orc, resident):
    """1.02 - (shift in x) converges by 1/1.02 per iteration: directions of one
    launch, of several, and of more than the resident form holds, where a
    launch per phase takes over."""
    lx, ly = 1500, 2
    n = lx * ly
    hop = np.zeros((4, n, 1, 1), dtype=complex)
    hop[0] = -1.0
    g = glx.StencilNc(lx, ly, 1, np.full((n, 1, 1), 1.02 + 0j), hop, None)
    h = glx.CStencilDev(g)
    rng = np.random.default_rng(5)
    b = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    nb = np.linalg.norm(b)

    def residual(x):
        x = x.reshape(ly, lx)
        return np.linalg.norm(b - (1.02 * x - np.roll(x, -1, axis=1)).reshape(-1))

    for stop, eps in ((64, 1e-10), (65, 1e-10), (130, 1e-10), (512, 1e-10), (513, 1e-10), (4000, 1e-6)):
        (x, i), (xl, il) = gcr_both(glx, resident, h, b, np.zeros(n, dtype=complex), max_iter=stop, eps=eps)
        print(stop, i.iter, il.iter, residual(x) / nb, flush=True)
        assert i.success == il.success and abs(i.iter - il.iter) <= (0 if stop < 600 else 2)
        assert abs(residual(x) - residual(xl)) <= (1e-8 if stop < 600 else 0.05) * residual(xl)
        assert abs(np.sqrt(i.resSq) - residual(x)) <= 1e-13 * nb
    assert i.success and i.iter > 520


def test_gcr_from_several_threads(glx, orc):
    """Solves of one kernel instance with different amounts of LDS (stencils
    of 5 and 13 terms and several colours), from several threads at once: the
    bits each gives alone."""
    work = [coarse(glx, orc, *s)[1:] for s in ((32, 32, 8, False), (24, 24, 6, True), (20, 24, 4, False), (9, 7, 12, True))]
    alone, got = [], [None] * len(work)
    for h, b, x0 in work:
        dx = glx.DeviceArray(x0)
        assert h.solve("gcr", dx, glx.DeviceArray(b), max_iter=400, eps=1e-10).success
        alone.append(dx.download())

    def run(k):
        h, b, x0 = work[k]
        db = glx.DeviceArray(b)
        for _ in range(40):
            dx = glx.DeviceArray(x0)
            h.solve("gcr", dx, db, max_iter=400, eps=1e-10)
            x = dx.download()
            if got[k] is None or np.array_equal(got[k], alone[k]):  # (the first that differs stays)
                got[k] = x

    ts = [threading.Thread(target=run, args=(k,)) for k in range(len(work))]
    with resident_solves(glx, 40 * len(work)):
        for t in ts:
            t.start()
        for t in ts:
            t.join()
    for a, g in zip(alone, got):
        assert np.array_equal(a, g)


def test_gcr_waits_that_run_out(glx, orc, resident):
    o, h, b, x0 = coarse(glx, orc, 32, 32, 8, False)
    resident(True, 1)
    dx = glx.DeviceArray(x0)
    with resident_solves(glx, 0, gave_up=1):
        assert h.solve("gcr", dx, glx.DeviceArray(b), max_iter=400, eps=1e-10).success
    assert np.linalg.norm(b - orc.cstencil_apply(o, dx.download())) <= 1.01e-10 * np.linalg.norm(b)


def test_guess_stop_and_zero(glx, orc):
    """A guess that is nearly the solution, max_iter stops, b = 0."""
    lx, ly, m = 130, 70, 0.1
    links, b, lat, db = system(glx, orc, lx, ly)
    kw = dict(links=links, mass=m, lx=lx, ly=ly)
    x0, _ = orc.solve("cg", "staggered_normal", b, None, max_iter=5000, eps=1e-6, **kw)
    xo, io = orc.solve("cg", "staggered_normal", b, x0, max_iter=5000, eps=1e-10, **kw)
    with resident_solves(glx, 8):
        dx = glx.DeviceArray(x0)
        ig = glx.dev_solve("cg", lat, "staggered_normal", m, dx, db, max_iter=5000)
        # (nearest: the serial sums round differently)
        assert abs(ig.iter - io.iter) <= 1 and relerr(dx.download(), xo) < 1e-9
        for stop in (1, 2, 7):
            xo, io = orc.solve("cg", "staggered_normal", b, None, max_iter=stop, eps=1e-10, **kw)
            dx = glx.DeviceArray(np.zeros_like(b))
            ig = glx.dev_solve("cg", lat, "staggered_normal", m, dx, db, max_iter=stop)
            assert (ig.iter, ig.success, ig.ops_count) == (io.iter, io.success, io.ops_count)
            assert relerr(dx.download(), xo) < 1e-12 and abs(ig.resSq - io.resSq) < 1e-10 * io.resSq
            dx.upload(np.zeros_like(b))
            im = glx.dev_cg_mixed(lat, "staggered_normal", m, dx, db, max_iter=stop)
            assert not im.success and im.iter == stop and relerr(dx.download(), xo) < 1e-4
        z = glx.DeviceArray(np.zeros_like(b))
        dx = glx.DeviceArray(np.zeros_like(b))
        im = glx.dev_cg_mixed(lat, "staggered_normal", m, dx, z)
        assert im.success and im.resSq == 0.0 and not dx.download().any()


def test_a_chosen_launch_form_is_taken(glx, orc):
    """A launch form set for the process or for the lattice's size keeps the
    mixed solve, even/odd included, in launches; another size's entry, the
    autotuner's and a removed one do not."""
    lx, ly, m = 256, 64, 0.1
    links, b, lat, db = system(glx, orc, lx, ly)

    def solves(n):
        for _ in range(2):
            dx = glx.DeviceArray(np.zeros_like(b))
            with resident_solves(glx, n):
                info = glx.dev_cg_mixed(lat, "staggered_normal", m, dx, db)
            r = b - orc.apply("staggered_normal", dx.download(), links, m, lx, ly)
            assert info.success and np.linalg.norm(r) <= 1.001e-10 * np.linalg.norm(b)
        with resident_solves(glx, n):
            assert glx.dev_solve_staggered_eo(lat, m, glx.DeviceArray(np.zeros_like(b)), db, "mixed")[0].success

    solves(1)
    try:
        for rows in (0, 8, 16):
            glx.set_sstep_rows(lx, ly, rows)
            solves(0)
        glx.set_sstep_rows(lx, ly, -1)
        for form in (0, 1):
            glx.set_sstep_form_entry(lx, ly, form)
            solves(0)
        glx.set_sstep_form_entry(lx, ly, -1)
        glx.set_sstep_rows(lx, 2 * ly, 8)
        solves(1)
        glx.set_sstep_rows(lx, ly, 8)
        glx.autotune_sstep(lat, reps=4)  # (replaces the entry)
        solves(1)
        glx.set_sstep_rows(lx, ly, 8)
        solves(0)
    finally:
        glx.set_sstep_rows(lx, ly, -1)
        glx.set_sstep_rows(lx, 2 * ly, -1)
        glx.set_sstep_form_entry(lx, ly, -1)
    solves(1)
    for s, rows in ((1, 0), (2, 8)):
        glx.set_sstep(s, rows)
        try:
            solves(0)
        finally:
            glx.set_sstep()


def test_waits_that_run_out(glx, orc, resident):
    """With a single poll per wait the launch gives up, and the solve runs with
    a launch per iteration: the same answer."""
    lx, ly, m = 130, 70, 0.1
    links, b, lat, db = system(glx, orc, lx, ly)
    xo, io = orc.solve("cg", "staggered_normal", b, None, links=links, mass=m, lx=lx, ly=ly, max_iter=5000, eps=1e-10)
    resident(True, 1)
    dx = glx.DeviceArray(np.zeros_like(b))
    with resident_solves(glx, 0, gave_up=1):
        ig = glx.dev_solve("cg", lat, "staggered_normal", m, dx, db, max_iter=5000)
    assert abs(ig.iter - io.iter) <= 1 and relerr(dx.download(), xo) < 1e-9
    dx.upload(np.zeros_like(b))
    with resident_solves(glx, 0, gave_up=1):
        assert glx.dev_cg_mixed(lat, "staggered_normal", m, dx, db).success
    assert relerr(dx.download(), xo) < 1e-9


def test_no_launch_waits_for_another(glx, orc):
    """Solves of 65 and 190 blocks, which an XCD would have 9 + 24 of for its
    32 CUs, from two threads over and over: none gives up."""
    m = 0.1
    work = [system(glx, orc, lx, ly) for lx, ly in ((290, 208), (600, 600))]

    def run(k):
        _, b, lat, db = work[k]
        for _ in range(100 if k == 0 else 50):
            glx.dev_cg_mixed(lat, "staggered_normal", m, glx.DeviceArray(np.zeros_like(b)), db)

    ts = [threading.Thread(target=run, args=(k,)) for k in range(2)]
    with resident_solves(glx, 150):
        for t in ts:
            t.start()
        for t in ts:
            t.join()


def test_threads_share_the_chip(glx, orc):
    """Solves from several host threads at once, together wanting more blocks
    than there are CUs, give the bits each gives alone."""
    m = 0.1
    work = [system(glx, orc, lx, ly) for lx, ly in ((700, 512), (330, 222), (512, 400), (256, 256))]
    alone, got = [], [None] * len(work)
    for _, b, lat, db in work:
        dx = glx.DeviceArray(np.zeros_like(b))
        glx.dev_cg_mixed(lat, "staggered_normal", m, dx, db)
        alone.append(dx.download())

    def run(k):
        _, b, lat, db = work[k]
        for _ in range(3):
            dx = glx.DeviceArray(np.zeros_like(b))
            glx.dev_cg_mixed(lat, "staggered_normal", m, dx, db)
            got[k] = dx.download()

    ts = [threading.Thread(target=run, args=(k,)) for k in range(len(work))]
    with resident_solves(glx, 3 * len(work)):
        for t in ts:
            t.start()
        for t in ts:
            t.join()
    for a, g in zip(alone, got):
        assert np.array_equal(a, g)
