"""GPU parity of the HIP coupled step against the FP64 CPU oracle, through the C-ABI.

Bars:
  * FP64 LBM part (fused pull collide/boundary/stream/injection): bit-identical to
    the oracle's restatement of LBM.cu:278-1353 on the same state, any number of steps;
  * FP64 initial equilibria and E field: bit-identical;
  * Poisson: FP64 relative max error <= 1e-13 against the oracle's odd-extension FFT
    solve (a different algorithm: x,y FFT plus tridiagonal z solve on the GPU);
    FP32S <= 2e-6;
  * coupled FP64 steps: rel-L2 on u, q (interior) and phi against the oracle.
"""
import os

import numpy as np
import pytest

import ehd_amd as E
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu

FIELDS = (O.RHO, O.Q, O.PHI, O.UX, O.UY, O.UZ, O.EX, O.EY, O.EZ)


def oracle_box(nx, ny, nz, T=200.0, C=10.0, lam=0.25, uw=0.0, exf=0.0, seed=1, amp=1e-3, mode="hydro",
               hydro_density=0):
    ob = O.Box(O.make_params(nx, ny, nz, T=T, M=10.0, C_=C, Fe=4000.0, lam=lam, uw=uw, exf=exf))
    ob.groups = dict(T=T, C_=C, M=10.0, Fe=4000.0)
    if mode == "hydro":
        ob.init_hydrostatic(seed, amp, hydro_density)
    else:
        ob.initialization()
    return ob


def gpu_box(ob, precision=E.FP64, init=True):
    p = ob.p
    params = E.make_params(p.nx, p.ny, p.nz, **ob.groups, lam=p.V, lam_c=p.VC, uw=p.uw, exf=p.exf,
                           precision=precision, init_mode=E.INIT_FIELDS)
    b = E.Box(params)
    if init:
        b.init(np.stack([ob[k] for k in FIELDS]))
    return b


def oracle_pops(ob):
    return ob[O.F0], ob[O.F1], ob[O.H0], ob[O.H1]


def assert_same(got, ref, what):
    if not np.array_equal(got, ref):
        diff = np.abs(got - ref)
        idx = np.unravel_index(np.argmax(diff), diff.shape)
        raise AssertionError(f"{what}: not bit-identical, max abs {diff.max():.3e} at {idx} "
                             f"({np.count_nonzero(diff)} of {diff.size} differ)")


def compare_pops(b, ob, what):
    f0, f1, h0, h1 = b.read_populations()
    rf0, rf1, rh0, rh1 = oracle_pops(ob)
    assert_same(f1, rf1, what + " f1")
    assert_same(h1, rh1, what + " h1")
    assert_same(f0, rf0, what + " f0")
    assert_same(h0, rh0, what + " h0")


def compare_macros(b, ob, what):
    g = b.read_fields(("rho", "q", "ux", "uy", "uz"))
    for name, key in (("rho", O.RHO), ("q", O.Q), ("ux", O.UX), ("uy", O.UY), ("uz", O.UZ)):
        assert_same(g[name], ob[key], f"{what} {name}")


def rel_l2(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("shape", [(8, 6, 7), (16, 12, 10), (64, 64, 32)])
def test_init_equilibrium_bitexact(shape):
    ob = oracle_box(*shape)
    ob.init_equilibrium()
    with gpu_box(ob) as b:
        compare_pops(b, ob, "init")


@pytest.mark.parametrize("hd", [0, 1])
def test_product_hydrostatic_init_matches_oracle(hd):
    nx, ny, nz = 16, 12, 10
    ob = oracle_box(nx, ny, nz, seed=5, amp=1e-3, hydro_density=hd)
    ob.init_equilibrium()
    p = E.make_params(nx, ny, nz, T=200.0, C_=10.0, lam=0.25, precision=E.FP64,
                      init_mode=E.INIT_HYDROSTATIC, seed=5, amp=1e-3, hydro_density=hd)
    with E.Box(p) as b:
        b.init()
        f = b.read_fields()
        for name, key in (("rho", O.RHO), ("q", O.Q), ("phi", O.PHI), ("ux", O.UX), ("uy", O.UY),
                          ("uz", O.UZ), ("ex", O.EX), ("ey", O.EY), ("ez", O.EZ)):
            assert np.allclose(f[name], ob[key], rtol=1e-14, atol=1e-14 * max(1.0, np.abs(ob[key]).max())), name
        compare_pops(b, ob, "hydrostatic init")


@pytest.mark.parametrize("pattern", [E.PERTURB_ROLLS, E.PERTURB_SQUARES, E.PERTURB_CROSS, E.PERTURB_HEXAGONS])
def test_pattern_init_matches_oracle(pattern):
    nx, ny, nz = 24, 20, 12
    ob = O.Box(O.make_params(nx, ny, nz, T=200.0, M=10.0, C_=10.0, Fe=4000.0, lam=0.25))
    ob.init_hydrostatic(3, 1e-3, 0, pattern)
    p = E.make_params(nx, ny, nz, T=200.0, C_=10.0, lam=0.25, precision=E.FP64,
                      init_mode=E.INIT_HYDROSTATIC, seed=3, amp=1e-3, pattern=pattern)
    with E.Box(p) as b:
        b.init()
        f = b.read_fields(("ux", "uy", "uz"))
        for name, key in (("ux", O.UX), ("uy", O.UY), ("uz", O.UZ)):
            assert np.abs(ob[key]).max() > 0 or name == "uy"
            assert np.allclose(f[name], ob[key], rtol=0, atol=1e-14 * max(1e-3, np.abs(ob[key]).max())), name


@pytest.mark.parametrize("precision", [E.FP64, E.FP32S])
def test_checkpoint_restart_bitexact(tmp_path, precision):
    """save_state/load_state restart the run bit for bit, also mid-run after
    the first (direct) step and across the E-buffer state."""
    ob = oracle_box(16, 12, 10)
    path = str(tmp_path / "state.ckpt")
    with gpu_box(ob, precision=precision) as a:
        a.step(3)
        a.save_state(path)
        a.step(5)
        ref = a.read_fields()
        ref_pops = a.read_populations()
        da = a.diagnostics()
    with gpu_box(ob, precision=precision, init=False) as b:
        b.load_state(path)
        b.step(5)
        got = b.read_fields()
        got_pops = b.read_populations()
        db = b.diagnostics()
    for k in ref:
        assert_same(got[k], ref[k], f"restart {k}")
    for g, r, n in zip(got_pops, ref_pops, ("f0", "f1", "h0", "h1")):
        assert_same(g, r, f"restart {n}")
    assert da.step == db.step and da.time == db.time
    with E.Box(E.make_params(16, 12, 12, precision=precision)) as c:
        with pytest.raises(E.EhdError):
            c.load_state(path)
    # same grid and precision, other physics: the populations (FP32S: stored
    # against the box's hydrostatic tables) would be wrong, so the load fails
    p = ob.p
    for other in (dict(T=201.0), dict(C_=11.0), dict(lam=0.2), dict(exf=1.0), dict(cfl=0.02)):
        kw = dict(T=200.0, C_=10.0, M=10.0, Fe=4000.0, lam=p.V, lam_c=p.VC, uw=p.uw, exf=p.exf)
        kw.update(other)
        with E.Box(E.make_params(16, 12, 10, precision=precision, init_mode=E.INIT_FIELDS, **kw)) as c:
            with pytest.raises(E.EhdError) as ei:
                c.load_state(path)
            assert ei.value.code == -1 and "differs" in str(ei.value), str(ei.value)


@pytest.mark.parametrize("case", [
    dict(shape=(8, 6, 7)),
    dict(shape=(16, 12, 10), lam=1.0 / 12.0),
    dict(shape=(12, 8, 9), uw=0.05, exf=40.0),
    dict(shape=(64, 64, 32)),
])
def test_lbm_steps_bitexact(case):
    """Three LBM steps (no Poisson in between: E stays the initial field)."""
    ob = oracle_box(*case["shape"], lam=case.get("lam", 0.25), uw=case.get("uw", 0.0), exf=case.get("exf", 0.0))
    ob.init_equilibrium()
    with gpu_box(ob) as b:
        for k in range(3):
            b.lbm_step()
            ob.stream_collide_save()
            compare_pops(b, ob, f"step {k + 1}")
            compare_macros(b, ob, f"step {k + 1}")


# States beyond 384 MB with rows that are no whole cache lines keep padded rows:
# 122 -> 128, 46 -> 48 doubles; 90 -> 96 floats.
@pytest.mark.parametrize("shape", [(122, 62, 64), (46, 120, 86)])
def test_lbm_steps_with_padded_rows_bitexact(shape):
    test_lbm_steps_bitexact(dict(shape=shape, uw=0.05, exf=40.0))


# A state that repeats along y does so on: a box of twice the rows, whose state is
# beyond 384 MB and keeps padded rows (90 -> 96, 252 -> 256 floats), steps as the box
# of one period does, which does not.  Whole potentials make the planes' means
# exact, so every value is the same bit for bit.
@pytest.mark.parametrize("shape", [(90, 76, 72), (252, 36, 56)])
def test_fp32s_steps_with_padded_rows_match_unpadded_bitwise(shape):
    nx, ny, nz = shape
    assert 432 * nx * ny * nz <= 384 << 20 < 2 * 432 * nx * ny * nz
    rng = np.random.default_rng(13)
    one = rng.standard_normal((9, nz, ny, nx))
    one[0] = 1600.0 + 1e-3 * one[0]
    one[1] = 1e-4 * np.abs(one[1])
    one[2] = rng.integers(0, 10000, (nz, ny, nx))
    one[3:6] *= 1e-3
    one[6:] *= 1e3
    fields, pops = [], []
    for f9 in (one, np.concatenate([one, one], axis=2)):
        p = E.make_params(nx, f9.shape[2], nz, T=200.0, lam=0.25, uw=0.05, exf=40.0, precision=E.FP32S,
                          init_mode=E.INIT_FIELDS)
        with E.Box(p) as b:
            b.init(f9)
            for _ in range(3):
                b.lbm_step()
            fields.append(b.read_fields())
            pops.append(b.read_populations())
    for k, v in fields[0].items():
        assert np.all(np.isfinite(v)), k
        assert_same(fields[1][k][:, :ny], v, f"{k}, first period")
        assert_same(fields[1][k][:, ny:], v, f"{k}, second period")
    for got, ref, n in zip(pops[1], pops[0], ("f0", "f1", "h0", "h1")):
        assert_same(got[..., :ny, :], ref, f"{n}, first period")
        assert_same(got[..., ny:, :], ref, f"{n}, second period")


@pytest.mark.parametrize("shape,precision,size", [((122, 62, 64), E.FP64, 8), ((90, 154, 70), E.FP32S, 4)])
def test_checkpoint_with_padded_rows_bitexact(tmp_path, shape, precision, size):
    """The file holds the same rows as an unpadded box's, and restarts bit for bit."""
    nx, ny, nz = shape
    S, path = nx * ny * nz, str(tmp_path / "state.ckpt")
    p = E.make_params(nx, ny, nz, T=200.0, precision=precision, pattern=E.PERTURB_SQUARES, amp=0.05)
    with E.Box(p) as a:
        a.init()
        a.step(2)
        a.save_state(path)
        saved = a.read_populations()
        a.step(2)
        ref, ref_pops = a.read_fields(), a.read_populations()
    # 2 x 26 populations, 3 rest arrays and 6 fields, the plane means, 3 doubles of E a node
    body = S * ((2 * 26 + 3 + 6) * size + 3 * 8) + nz * 8
    header = os.path.getsize(path) - body
    assert 0 < header < 256
    if precision == E.FP64:   # f of the state file: post-collision rows [z][y][d-1][x]; a pull along +x is d = 1
        rows = np.fromfile(path, dtype=np.float64, count=26 * S, offset=header).reshape(nz, ny, 26, nx)
        assert_same(np.roll(rows[:, :, 0, :], 1, axis=2), saved[1][0], "f_1 in the file")
    with E.Box(p) as b:
        b.load_state(path)
        b.step(2)
        got, got_pops = b.read_fields(), b.read_populations()
    for k in ref:
        assert_same(got[k], ref[k], f"restart {k}")
    for g, r, n in zip(got_pops, ref_pops, ("f0", "f1", "h0", "h1")):
        assert_same(g, r, f"restart {n}")


def test_reference_initial_state_bitexact():
    """gpu_initialization state (q=0, linear phi, E=0) through two LBM steps."""
    ob = oracle_box(12, 10, 8, mode="reference")
    ob.init_equilibrium()
    p = E.make_params(12, 10, 8, **ob.groups, lam=0.25, precision=E.FP64, init_mode=E.INIT_REFERENCE)
    with E.Box(p) as b:
        b.init()
        compare_pops(b, ob, "reference init")
        for k in range(2):
            b.lbm_step()
            ob.stream_collide_save()
            compare_pops(b, ob, f"reference step {k + 1}")


def test_lbm_with_phi_stencil_bitexact():
    """E = -grad(phi) computed inside the fused kernel equals efield() + collide."""
    ob = oracle_box(16, 12, 10)
    ob.init_equilibrium()
    with gpu_box(ob) as b:
        b.lbm_step()
        ob.stream_collide_save()
        ob.poisson()
        b.write_phi(ob[O.PHI])
        ob.efield()
        e = b.read_fields(("ex", "ey", "ez"))
        assert_same(e["ex"], ob[O.EX], "ex")
        assert_same(e["ey"], ob[O.EY], "ey")
        assert_same(e["ez"], ob[O.EZ], "ez")
        for k in range(2):
            b.lbm_step()
            ob.stream_collide_save()
            compare_pops(b, ob, f"phi step {k + 1}")
            compare_macros(b, ob, f"phi step {k + 1}")


def test_random_population_state_bitexact():
    """Arbitrary (non-equilibrium) populations written through the C-ABI."""
    ob = oracle_box(10, 8, 9)
    rng = np.random.default_rng(7)
    w = O.tables()["w"]
    shp = ob.shape
    ob[O.F0][...] = w[0] * 1600 * (1 + 1e-3 * rng.standard_normal(shp))
    ob[O.H0][...] = w[0] * 5 * (1 + 0.1 * rng.standard_normal(shp))
    for d in range(1, 27):
        ob[O.F1][d - 1] = w[d] * 1600 * (1 + 1e-3 * rng.standard_normal(shp))
        ob[O.H1][d - 1] = w[d] * 5 * (1 + 0.1 * rng.standard_normal(shp))
    with gpu_box(ob) as b:
        b.write_populations(*oracle_pops(ob))
        compare_pops(b, ob, "written")
        for k in range(2):
            b.lbm_step()
            ob.stream_collide_save()
            compare_pops(b, ob, f"random step {k + 1}")


@pytest.mark.parametrize("shape", [(8, 6, 7), (48, 48, 32), (80, 80, 12), (64, 64, 32), (122, 122, 10), (96, 96, 8),
                                   (64, 48, 200), (128, 128, 65), (16, 8, 300),
                                   # the compile-time plans of the bench box and of the largest configuration
                                   (256, 256, 34), (256, 256, 128), (512, 512, 12), (512, 512, 40)])
@pytest.mark.parametrize("precision", [E.FP64, E.FP32S])
def test_poisson_vs_oracle(shape, precision):
    nx, ny, nz = shape
    ob = oracle_box(nx, ny, nz)
    rng = np.random.default_rng(nx + nz)
    q = ob[O.Q] * (1 + 0.2 * rng.standard_normal(ob.shape))
    ob[O.Q][...] = q
    with gpu_box(ob, precision=precision) as b:
        b.write_charge(q)
        b.poisson()
        phi = b.read_fields(("phi",))["phi"]
    ob.poisson()
    err = np.max(np.abs(phi - ob[O.PHI])) / np.max(np.abs(ob[O.PHI]))
    tol = 1e-13 if precision == E.FP64 else 2e-6
    print(f"poisson {shape} prec={precision}: max rel err {err:.3e}")
    assert err < tol


# The runtime-planned transforms: each radix (2..5, 7, 9, 11, 13, 16), a prime
# stage alone, first and second (17, 61, 17 * 19), one side planned at compile
# time and the other not, a last block of rows that is not full, one row pair.
@pytest.mark.parametrize("shape", [(122, 122, 9), (34, 4, 6), (646, 2, 5), (64, 34, 7), (90, 154, 6), (18, 26, 11),
                                   (22, 98, 8), (112, 48, 5), (2, 14, 12), (200, 36, 6),
                                   # planes on both sides of the one-launch transforms' limit, and their plans
                                   (62, 66, 6), (64, 66, 6), (32, 32, 9), (32, 128, 5), (32, 130, 5)])
@pytest.mark.parametrize("precision", [E.FP64, E.FP32S])
def test_poisson_runtime_plans_vs_oracle(shape, precision):
    test_poisson_vs_oracle(shape, precision)


# The one-launch transforms of small planes give the separate passes' bits (debug
# level 2 runs those): squares with a compile-time plan, pairs of runtime plans of
# every radix (2..5, 7, 9, 11, 13, 16, a prime stage), and planes of which only
# one side, or each side another, has a compile-time plan.
@pytest.mark.parametrize("shape", [(32, 32), (64, 64), (48, 48), (36, 36), (24, 40), (2, 14), (18, 26), (22, 98),
                                   (62, 62), (34, 38), (16, 20), (58, 62), (32, 64), (64, 32), (48, 32), (80, 48),
                                   (32, 100), (64, 40), (64, 62), (16, 256), (32, 128)])
@pytest.mark.parametrize("precision", [E.FP64, E.FP32S])
def test_plane_transforms_match_the_passes_bitwise(shape, precision):
    nx, ny, nz = *shape, 9
    q = np.random.default_rng(7).standard_normal((nz, ny, nx))
    phi = []
    for level in (0, 1, 2):
        with E.Box(E.make_params(nx, ny, nz, T=200.0, precision=precision)) as b:
            b.init()
            b.set_debug_sync(level)
            b.write_charge(q)
            b.poisson()
            phi.append(b.read_fields(("phi",))["phi"])
    assert np.all(np.isfinite(phi[0])) and np.ptp(phi[0]) > 0
    assert_same(phi[1], phi[0], "checked after every launch")
    assert_same(phi[2], phi[0], "every transform in a launch of its own")


def test_diagnostics_current_vs_oracle():
    ob = oracle_box(16, 12, 10)
    ob.init_equilibrium()
    with gpu_box(ob) as b:
        b.step(3)
        ob.step(3)
        d = b.diagnostics()
        ref = ob.current()
        assert abs(d.current / ref - 1) < 1e-11, (d.current, ref)
        q = ob[O.Q][1:-1]
        assert abs(d.total_charge / (q.sum() * ob.p.dx ** 3) - 1) < 1e-12
        # umax = record_umax (LBM.cu:1673-1713) of the box's own uz, exactly;
        # the oracle's uz differs in the last bits (its Poisson is another
        # algorithm), so against it the bar is relative
        uz = b.read_fields(("uz",))["uz"]
        uz[-1] = 2 * uz[-2] - uz[-3]
        assert d.umax == max(0.0, uz.max())
        uo = ob[O.UZ].copy()
        uo[-1] = 2 * uo[-2] - uo[-3]
        assert abs(d.umax / max(0.0, uo.max()) - 1) < 1e-12
        assert d.step == 3


# Field reads below and above one megabyte (with and without worker threads), with
# a last piece that is not full, and with more pieces than staging slots.
@pytest.mark.parametrize("shape", [(16, 12, 10), (64, 64, 33), (122, 62, 40), (256, 256, 44)])
@pytest.mark.parametrize("precision", [E.FP64, E.FP32S])
def test_field_reads_are_exact(shape, precision):
    nx, ny, nz = shape
    rng = np.random.default_rng(5)
    q, phi = rng.standard_normal((2, nz, ny, nx))
    with E.Box(E.make_params(nx, ny, nz, T=200.0, precision=precision)) as b:
        b.init()
        b.step(2)
        b.write_charge(q)
        b.write_phi(phi)
        every = b.read_fields()
        alone = {k: b.read_fields((k,))[k] for k in every}
    for k, v in every.items():
        assert np.array_equal(v, alone[k]), k
    assert np.array_equal(every["q"], q if precision == E.FP64 else q.astype(np.float32).astype(np.float64))
    # FP32S keeps phi as a float beside its plane's mean: rounded once
    assert np.max(np.abs(every["phi"] - phi)) <= (0.0 if precision == E.FP64 else 2.0**-23 * np.max(np.abs(phi)))


def test_profile_sampling_counts_launches():
    """ehd_profile_enable(b, n) brackets the LBM launch and the Poisson chain
    of the steps whose index is a multiple of n, and every ehd_step call; the
    sampled steps compute exactly what unsampled ones do."""
    ob = oracle_box(16, 12, 10)
    ob.init_equilibrium()
    with gpu_box(ob) as b, gpu_box(ob) as ref:
        b.profile_enable(True, every=4)
        b.step(12)            # steps 0..11: 0, 4, 8 sampled
        b.step(5)             # steps 12..16: 12, 16
        pr = b.profile_read()
        assert (pr.lbm_launches, pr.poisson_calls, pr.steps) == (5, 5, 2), pr
        assert pr.lbm_ms > 0 and pr.poisson_ms > 0 and pr.step_ms > pr.lbm_ms
        ref.step(17)
        got, want = b.read_fields(("q", "uz")), ref.read_fields(("q", "uz"))
        for k in ("q", "uz"):
            assert_same(got[k], want[k], k)
        with pytest.raises(E.EhdError):
            b.profile_enable(True, every=-1)


def test_nusselt_reference_and_steady_detector():
    """Nu = I / I_hs.  With the analytic reference Nu is 1 on the hydrostatic
    start.  The lattice's own no-flow steady current (a 2x2 column run to
    steady) equals the oracle's, and a box below the convection threshold
    relaxes to it: the detector then reports Nu = 1."""
    p = E.make_params(16, 16, 17, T=50.0, C_=10.0, lam=0.25, precision=E.FP64, init_mode=E.INIT_HYDROSTATIC,
                      seed=4, amp=1e-4)
    ob = O.Box(O.make_params(2, 2, 17, T=50.0, M=10.0, C_=10.0, Fe=4000.0, lam=0.25))
    ob.init_hydrostatic(1, 0.0, 0)
    ob.init_equilibrium()
    ob.step(45000)
    with E.Box(p) as b:
        b.init()
        d0 = b.diagnostics()
        assert abs(d0.nusselt - 1.0) < 1e-12, d0.nusselt
        ihs = b.hydrostatic_reference(check_every=500, tol=1e-10)
        ref = ob.current() * (16 * 16 / 4)
        print(f"discrete hydrostatic current {ihs:.12g}, oracle {ref:.12g}, analytic {d0.current:.12g}")
        assert abs(ihs / ref - 1) < 1e-6
        s = b.run_to_steady(check_every=500, tol=1e-8, max_steps=60000)
        print(f"steady after {s.steps} steps: Nu {s.nusselt:.10f} delta {s.delta:.2e}")
        assert s.converged == 1 and s.delta < 1e-8
        assert abs(s.nusselt - 1.0) < 1e-5
        d1 = b.diagnostics()
        assert d1.step == s.steps and d1.nusselt == s.nusselt


def _coupled_errors(ga, ob):
    """rel-L2 of u, q (interior) and phi of a field dict or oracle box against the oracle box ob."""
    def get(src, key, name):
        return src[name] if isinstance(src, dict) else src[key]
    u_a = np.stack([get(ga, O.UX, "ux"), get(ga, O.UY, "uy"), get(ga, O.UZ, "uz")])[:, 1:-1]
    u_b = np.stack([ob[O.UX], ob[O.UY], ob[O.UZ]])[:, 1:-1]
    return {"u": rel_l2(u_a, u_b), "q": rel_l2(get(ga, O.Q, "q")[1:-1], ob[O.Q][1:-1]),
            "phi": rel_l2(get(ga, O.PHI, "phi"), ob[O.PHI])}


def test_coupled_fp64_config1_vs_oracle():
    """64x64x32, T=200, C=10, M=10, Fe=4000, Lambda=1/4, hydrostatic charge and potential,
    uniform rho0, 1e-3 velocity noise; 1000 coupled FP64 steps on the GPU and in the oracle,
    compared (and held to the bar) every 100 steps.

    Bar: phi and q within 1e-12 rel-L2.  For u the bar is 1e-12 or the FP64 floor of this
    problem, whichever is larger: the floor is the distance between two FP64 evaluations
    of the same discrete step inside the oracle (odd-extension FFT Poisson, step, vs x,y FFT
    plus tridiagonal z solve, step_tridiag), on the same start.  The GPU must not be farther
    than twice that floor from either: from the FFT leg, which restates the reference, and
    from the tridiagonal leg, whose algorithm the GPU shares."""
    ob = oracle_box(64, 64, 32)
    ob.init_equilibrium()
    ot = oracle_box(64, 64, 32)
    ot.init_equilibrium()
    with gpu_box(ob) as b:
        for k in range(1, 11):
            b.step(100)
            ob.step(100)
            ot.step_tridiag(100)
            g = b.read_fields(("q", "phi", "ux", "uy", "uz"))
            errs, tri, floor = _coupled_errors(g, ob), _coupled_errors(g, ot), _coupled_errors(ot, ob)
            print(f"step {100 * k}: GPU vs FFT oracle {errs}; GPU vs tridiagonal oracle {tri}; "
                  f"oracle floor {floor}", flush=True)
            for e in (errs, tri):     # the bar at every checkpoint of the trajectory
                assert e["phi"] < 1e-12 and e["q"] < 1e-12, (100 * k, e, floor)
                assert e["u"] < max(1e-12, 2.0 * floor["u"]), (100 * k, e, floor)


@pytest.mark.timeout(400)
def test_coupled_fp64_reference_configuration():
    """The reference's own configuration (LBM.h:31-86): 122x122x101, T ~ 996,
    M = C = 10, Fe = 4000, Lambda = 1/12, Lambda_c = 1e-6, from the reference
    initial state (rho0, q = 0, linear phi, u = 0, E = 0; LBM.cu:69-96);
    300 coupled FP64 steps on the GPU and in the oracle (the charge front
    leaves the injection wall).  Bar: q, phi within 1e-12 rel-L2, u within
    1e-12 or twice the oracle's own FP64 floor (FFT vs tridiagonal Poisson)."""
    dp = E.default_params()
    nx, ny, nz, nsteps = dp.nx, dp.ny, dp.nz, 300
    op = O.make_params(nx, ny, nz, T=dp.T, M=dp.M, C_=dp.C, Fe=dp.Fe, lam=dp.lambda_f, lam_c=dp.lambda_c)
    ob = O.Box(op)
    ob.initialization()
    ob.init_equilibrium()
    with E.Box(dp) as b:
        b.init()
        compare_pops(b, ob, "reference configuration init")
        b.step(nsteps)
        g = b.read_fields(("q", "phi", "ux", "uy", "uz"))
    ob.step(nsteps)
    ot = O.Box(op)
    ot.initialization()
    ot.init_equilibrium()
    ot.step_tridiag(nsteps)
    errs, tri, floor = _coupled_errors(g, ob), _coupled_errors(g, ot), _coupled_errors(ot, ob)
    print(f"122x122x101 reference configuration, {nsteps} steps: GPU vs FFT oracle {errs}; "
          f"GPU vs tridiagonal oracle {tri}; oracle floor {floor}; q max {np.abs(ob[O.Q]).max():.4g}")
    assert np.abs(ob[O.Q][1:-1]).max() > 0
    for e in (errs, tri):
        assert e["phi"] < 1e-12 and e["q"] < 1e-12, (e, floor)
        assert e["u"] < max(1e-12, 2.0 * floor["u"]), (e, floor)


@pytest.mark.parametrize("hd", [0, 1])
def test_fp32s_vs_fp64_short(hd):
    """FP32 storage of shifted populations against the FP64 path, same start."""
    ob = oracle_box(32, 32, 16, hydro_density=hd)
    ob.init_equilibrium()
    res = {}
    for prec in (E.FP64, E.FP32S):
        with gpu_box(ob, precision=prec) as b:
            b.step(300)
            res[prec] = b.read_fields(("q", "phi", "ux", "uy", "uz"))
    a, r = res[E.FP32S], res[E.FP64]
    errs = {k: rel_l2(a[k][1:-1], r[k][1:-1]) for k in ("q", "phi", "ux", "uy", "uz")}
    print(f"FP32S vs FP64 after 300 steps (hydro_density={hd}): {errs}")
    assert errs["q"] < 1e-5 and errs["phi"] < 1e-5
    assert max(errs["ux"], errs["uy"], errs["uz"]) < 1e-2


def _nine(f):
    return np.stack([f[k] for k in ("rho", "q", "phi", "ux", "uy", "uz", "ex", "ey", "ez")])


def _field_errors(a, r):
    u_a = np.stack([a["ux"], a["uy"], a["uz"]])[:, 1:-1]
    u_r = np.stack([r["ux"], r["uy"], r["uz"]])[:, 1:-1]
    return {"q": rel_l2(a["q"][1:-1], r["q"][1:-1]), "phi": rel_l2(a["phi"], r["phi"]), "u": rel_l2(u_a, u_r)}


def _fp32s_vs_fp64(params_of, fields9, nsteps):
    """Run the same start in both precisions; errors of fields, Nu and current,
    the FP64 diagnostics and both field sets."""
    out = {}
    for prec in (E.FP64, E.FP32S):
        with E.Box(params_of(prec)) as b:
            b.init(fields9)
            b.step(nsteps)
            out[prec] = (b.read_fields(("q", "phi", "ux", "uy", "uz")), b.diagnostics())
    (a, da), (r, dr) = out[E.FP32S], out[E.FP64]
    errs = dict(_field_errors(a, r), Nu=abs(da.nusselt / dr.nusselt - 1), current=abs(da.current / dr.current - 1))
    return errs, dr, a, r


def test_fp32s_vs_fp64_developed_convection():
    """A developed convecting state (64x64x64, T=300, C=10, grown from noise,
    Nu ~ 1.8, velocities ~6x the drift velocity): the FP32S path against the
    FP64 path (which is bit-identical to the oracle's step) over 20,000
    further steps from the same fields.  Here the populations stray far from
    the hydrostatic shift, so their float rounding is relative to the
    convective part itself; the two paths settle to steady states that differ
    by ~1e-4 in the fields and ~4e-5 in Nu.  Bar: Nu and the current within
    0.1 %, the fields within 2e-4 rel-L2."""
    def params_of(prec, init=E.INIT_FIELDS):
        return E.make_params(64, 64, 64, T=300.0, C_=10.0, lam=0.25, precision=prec, init_mode=init, seed=11,
                             amp=1e-3, cfl=0.04)
    with E.Box(params_of(E.FP32S, E.INIT_HYDROSTATIC)) as b:
        b.init()
        b.step(120000)
        start = _nine(b.read_fields())
    errs, dr, _, _ = _fp32s_vs_fp64(params_of, start, 20000)
    print(f"developed convection, FP64 Nu {dr.nusselt:.6f}; FP32S vs FP64 after 20000 steps: {errs}")
    assert dr.nusselt > 1.5
    assert errs["Nu"] < 1e-3 and errs["current"] < 1e-3, errs
    assert max(errs["u"], errs["q"], errs["phi"]) < 2e-4, errs


def _fp32s_vs_fp64_checkpoints(params_of, nsteps, every, what):
    """Both precisions from the same start (the FP64 path's hydrostatic start
    with its seeded noise), compared every `every` steps.  At every
    checkpoint: q and phi within 1e-5 rel-L2, Nu and current within 0.1 %, and
    u within 1e-5 of the run's velocity scale, ||u_FP32S - u_FP64|| /
    max over checkpoints of ||u_FP64||.  Most of u in these starts is a
    plane-uniform standing acoustic wave (the start is not the discrete
    equilibrium under the force); where it passes through zero ||u|| drops
    ~1000-fold, and the instantaneous rel-L2 of u -- for two schemes whose
    waves differ in phase by d, about d tan(wt) -- has no bound there.  The
    instantaneous u error is printed at every checkpoint as well."""
    with E.Box(params_of(E.FP64, E.INIT_HYDROSTATIC)) as b:
        b.init()
        start = _nine(b.read_fields())
    rows = []
    with E.Box(params_of(E.FP64)) as r, E.Box(params_of(E.FP32S)) as a:
        r.init(start)
        a.init(start)
        for k in range(every, nsteps + 1, every):
            r.step(every)
            a.step(every)
            fr = r.read_fields(("q", "phi", "ux", "uy", "uz"))
            fa = a.read_fields(("q", "phi", "ux", "uy", "uz"))
            dr, da = r.diagnostics(), a.diagnostics()
            ur = np.stack([fr["ux"], fr["uy"], fr["uz"]])[:, 1:-1]
            ua = np.stack([fa["ux"], fa["uy"], fa["uz"]])[:, 1:-1]
            errs = dict(_field_errors(fa, fr), Nu=abs(da.nusselt / dr.nusselt - 1),
                        current=abs(da.current / dr.current - 1))
            rows.append((k, errs, float(np.linalg.norm(ua - ur)), float(np.linalg.norm(ur)), dr.umax))
    uscale = max(r[3] for r in rows)
    for k, errs, du, nu, umax in rows:
        errs["u_scale"] = du / uscale
        print(f"{what} step {k}: umax {umax:.3e} |u|/max|u| {nu / uscale:.2e} "
              + " ".join(f"{n} {v:.2e}" for n, v in errs.items()), flush=True)
    for k, errs, du, nu, umax in rows:
        assert errs["u_scale"] < 1e-5 and errs["q"] < 1e-5 and errs["phi"] < 1e-5, (k, errs)
        assert errs["Nu"] < 1e-3 and errs["current"] < 1e-3, (k, errs)
    return rows


@pytest.mark.timeout(400)   # ~60 s
def test_fp32s_vs_fp64_256x256x128_20000_steps():
    """Config 2: the bench box's own start (256x256x128, T=400, C=10,
    hydrostatic q and phi, uniform rho0, 1e-3 velocity noise from seed 2)
    stepped 20,000 times in both precisions, the bar held at every 1,000-step
    checkpoint.  The start is not the discrete equilibrium under the force,
    so a plane-uniform acoustic wave carries most of u (umax swings between
    ~5e-2 and ~1e-4)."""
    def params_of(prec, init=E.INIT_FIELDS):
        return E.make_params(256, 256, 128, T=400.0, C_=10.0, lam=0.25, precision=prec, init_mode=init, seed=2,
                             amp=1e-3)
    _fp32s_vs_fp64_checkpoints(params_of, 20000, 1000, "256x256x128")


@pytest.mark.timeout(600)   # ~150 s
def test_fp32s_vs_fp64_512x512x128():
    """Config 5: the largest configuration (512x512x128, 33.5 M nodes; T=1000,
    C=10, hydrostatic start + 1e-3 noise from seed 5) over its full 10,000
    steps in both precisions, the bar held at every 1,000-step checkpoint."""
    def params_of(prec, init=E.INIT_FIELDS):
        return E.make_params(512, 512, 128, T=1000.0, C_=10.0, lam=0.25, precision=prec, init_mode=init, seed=5,
                             amp=1e-3)
    _fp32s_vs_fp64_checkpoints(params_of, 10000, 1000, "512x512x128")


def test_fp32s_vs_fp64_256x256x128():
    """The bench box (256x256x128, T=400, C=10) started from hydrostatic q and
    phi with roll velocities of 20 % of the drift velocity: 1000 steps in both
    precisions.  Bar: u, q, phi within 1e-5 rel-L2, Nu and current within 0.1 %."""
    def params_of(prec, init=E.INIT_FIELDS):
        return E.make_params(256, 256, 128, T=400.0, C_=10.0, lam=0.25, precision=prec, init_mode=init, seed=2,
                             amp=0.05, pattern=E.PERTURB_ROLLS)
    with E.Box(params_of(E.FP64, E.INIT_HYDROSTATIC)) as b:
        b.init()
        start = _nine(b.read_fields())
    errs, dr, _, _ = _fp32s_vs_fp64(params_of, start, 1000)
    print(f"256x256x128, FP64 Nu {dr.nusselt:.6f}; FP32S vs FP64 after 1000 steps: {errs}")
    assert errs["u"] < 1e-5 and errs["q"] < 1e-5 and errs["phi"] < 1e-5, errs
    assert errs["Nu"] < 1e-3 and errs["current"] < 1e-3, errs
