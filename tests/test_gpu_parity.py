"""HIP path against the reference's golden vectors and the CPU oracle.

Every test calls the GPU library through its C ABI (libludwig_hip.so via
ludwig_amd).  The bar for FP64 is bit-exact equality (the kernels are built
with -ffp-contract=off and keep the reference's operation order).
"""

import hashlib

import numpy as np
import pytest

import ludwig_amd as L
import oracle as O

pytestmark = pytest.mark.gpu


def sha(a):
    return hashlib.sha256(np.ascontiguousarray(a, dtype="<f8").tobytes()).hexdigest()


def assert_exact(got, want, what):
    got, want = np.asarray(got), np.asarray(want)
    assert got.shape == want.shape, what
    bad = np.flatnonzero(got != want)
    if bad.size:
        i = bad[0]
        rel = np.max(np.abs(got - want) / np.maximum(np.abs(want), 1e-300))
        pytest.fail(f"{what}: {bad.size}/{got.size} differ, first {i}: {got[i]!r} vs {want[i]!r}; max rel {rel:.3e}")


@pytest.mark.parametrize("case,relax,tau", [
    ("collide_m10", L.M10, 0.8), ("collide_bgk", L.BGK, 0.8),
    ("collide_trt", L.TRT, 0.8), ("collide_m10_tau1", L.M10, 1.0)])
def test_collide_golden(golden, case, relax, tau):
    g = golden(case)
    n = int(g["n"])
    print(f"case {case} n={n}", flush=True)
    s = L.SingleFluid((n, n, n), tau=tau, relax=relax)
    s.set_f(g["f_in"])
    s.set_hydro(force=g["force"])
    s.u_zero()
    s.collide()
    assert_exact(s.f(), g["f_out"], "f")
    rho, u, _ = s.hydro_fields()
    assert_exact(rho, g["rho"], "rho")
    assert_exact(u, g["u"], "u")
    s.close()


def test_propagation_golden(golden):
    g = golden("prop")
    n = int(g["n"])
    s = L.SingleFluid((n, n, n), tau=0.8)
    s.set_f(g["f_in"])
    s.propagate()
    assert_exact(s.f(), g["f_out"], "f after one propagation")
    # a second propagation without collision materialises the first
    s.propagate()
    assert_exact(s.f(), O.propagate((n, n, n), g["f_out"]), "f after two propagations")
    s.close()


def _gm(g):
    return tuple(float(v) for v in g["grad_mu"]) if "grad_mu" in g else (0.0, 0.0, 0.0)


@pytest.mark.parametrize("case,method", [("force_stress", L.FORCE_STRESS_DIVERGENCE),
                                         ("force_gradmu", L.FORCE_PHI_GRADMU),
                                         ("force_gradmu_ext", L.FORCE_PHI_GRADMU)])
def test_force_golden(golden, case, method):
    """force_gradmu_ext: an external chemical potential gradient adds
    -phi grad_mu to the phi grad mu force (phi_grad_mu.c:123-160)."""
    g = golden(case)
    n = int(g["n"])
    args = [str(a) for a in g["args"]]
    a, b_, k = map(float, args[4:7])
    print(f"case {case}", flush=True)
    b = L.BinaryFluid((n, n, n), a=a, b=b_, kappa=k, tau=1.0, force_method=method, grad_mu=_gm(g))
    b.set_phi(g["phi"])
    b.f_zero()
    b.force_stage()
    _, _, F = b.hydro_fields()
    assert_exact(F, g["force"], "force")
    b.close()


@pytest.mark.parametrize("case,method", [("force27_stress", L.FORCE_STRESS_DIVERGENCE),
                                         ("force27_gradmu", L.FORCE_PHI_GRADMU)])
def test_force27_golden(golden, case, method):
    """The 27-point gradient (gradient_3d_27pt_fluid.c) through the force."""
    g = golden(case)
    n = int(g["n"])
    args = [str(a) for a in g["args"]]
    a, b_, k = map(float, args[4:7])
    b = L.BinaryFluid((n, n, n), a=a, b=b_, kappa=k, tau=1.0, force_method=method, stencil=27)
    b.set_phi(g["phi"])
    b.f_zero()
    b.force_stage()
    _, _, F = b.hydro_fields()
    assert_exact(F, g["force"], "force")
    b.close()


def _host_fed_str(phi, grad, delsq, a, b, kappa):
    """fe_symm_fed and fe_symm_str (symmetric.c:285-299, 334-362) in the
    reference's operation order, elementwise in IEEE double."""
    gg = grad[0] * grad[0] + grad[1] * grad[1] + grad[2] * grad[2]
    fed = (0.5 * a + 0.25 * b * phi * phi) * phi * phi + 0.5 * kappa * gg
    p0 = 0.5 * a * phi * phi + 0.75 * b * phi * phi * phi * phi - kappa * phi * delsq - 0.5 * kappa * gg
    st = np.empty((9,) + phi.shape)
    for i in range(3):
        for j in range(3):
            st[3 * i + j] = p0 * float(i == j) + kappa * grad[i] * grad[j]
    return fed, st


@pytest.mark.parametrize("case,stencil", [("force_stress", 7), ("force27_stress", 27),
                                          ("force_gradmu", 7)])
def test_gradient_and_mu_readback_golden(golden, case, stencil):
    """After field_grad_compute(), the host read-back the reference's
    statistics use (field_grad_memcpy, field_grad_scalar_grad/_delsq,
    fe_symm_mu; field_grad.c:319-339, symmetric.c:308-318) equals the
    reference's grad, delsq and mu bit for bit; fe_symm_fed/_str equal the
    reference's formulas evaluated on those."""
    g = golden(case)
    n = int(g["n"])
    args = [str(a) for a in g["args"]]
    a, b_, k = map(float, args[4:7])
    print(f"case {case}", flush=True)
    b = L.BinaryFluid((n, n, n), a=a, b=b_, kappa=k, tau=1.0, stencil=stencil)
    b.set_phi(g["phi"])
    b.gradient_stage()
    grad, delsq, mu, fed, st = b.gradient_readback()
    assert_exact(grad.ravel(), g["grad"], "grad")
    assert_exact(delsq, g["delsq"], "delsq")
    assert_exact(mu, g["mu"], "mu")
    fed_ref, st_ref = _host_fed_str(g["phi"], g["grad"].reshape(3, -1), g["delsq"], a, b_, k)
    assert_exact(fed, fed_ref, "fed")
    assert_exact(st.ravel(), st_ref.ravel(), "str")
    # the read-back after a force calculation on the same phi is the same
    b.f_zero()
    b.force_stage()
    grad2, delsq2, mu2, _, _ = b.gradient_readback()
    assert_exact(grad2.ravel(), g["grad"], "grad after force")
    assert_exact(mu2, g["mu"], "mu after force")
    b.close()


@pytest.mark.parametrize("case,order", [("ch_order1", 1), ("ch_order2", 2), ("ch_order3", 3),
                                        ("ch_order4", 4), ("ch_order5", 5), ("ch_gradmu_o2", 2)])
def test_cahn_hilliard_golden(golden, case, order):
    """Advection orders 1-5 and the external gradient on the face fluxes."""
    g = golden(case)
    n = int(g["n"])
    args = [str(a) for a in g["args"]]
    a, b_, k, m = map(float, args[4:8])
    print(f"case {case}", flush=True)
    b = L.BinaryFluid((n, n, n), a=a, b=b_, kappa=k, mobility=m, tau=1.0, order=order, grad_mu=_gm(g))
    b.set_phi(g["phi_in"])
    b.set_hydro(u=g["u"])
    b.cahn_hilliard_stage()
    assert_exact(b.phi_field(), g["phi_out"], "phi")
    b.close()


def _binary_args(g):
    args = [str(a) for a in g["args"]]
    n, nsteps, seed, order = int(args[1]), int(args[2]), int(args[3]), int(args[4])
    a, b, k, m, tau, phi0, amp = map(float, args[5:12])
    return n, nsteps, seed, order, a, b, k, m, tau, phi0, amp


@pytest.mark.parametrize("case", ["binary16_o1_s20", "binary16_o3_s10", "binary16_o2_s5",
                                  "binary16_g27_s10", "binary16_g27_o3_s10",
                                  "binary16_o4_s10", "binary16_o5_s10",
                                  "binary16_gmu_s10", "binary16_gmu_stress_s10"])
def test_binary_step_golden(golden, case):
    """Whole steps: order 4 through the single-pass step kernel, order 5
    through the staged kernels; grad_mu with both force methods."""
    g = golden(case)
    n, nsteps, seed, order, a, b_, k, m, tau, phi0, amp = _binary_args(g)
    stencil = int(g["stencil"]) if "stencil" in g else 7
    gradmu = "force_method" in g and int(g["force_method"]) == 1
    method = L.FORCE_PHI_GRADMU if gradmu else L.FORCE_STRESS_DIVERGENCE
    print(f"case {case}", flush=True)
    b = L.BinaryFluid((n, n, n), a=a, b=b_, kappa=k, mobility=m, order=order, tau=tau,
                      stencil=stencil, force_method=method, grad_mu=_gm(g))
    b.init_spinodal(seed, phi0, amp)
    if "phi_init" in g:
        assert_exact(b.phi_field(), g["phi_init"], "phi_init")
    if "phi_10" in g:
        b.step(10)
        assert_exact(b.phi_field(), g["phi_10"], "phi at step 10")
        b.step(nsteps - 10)
    else:
        b.step(nsteps)
    assert_exact(b.phi_field(), g["phi"], "phi")
    rho, u, _ = b.hydro_fields()
    assert_exact(rho, g["rho"], "rho")
    assert_exact(u, g["u"], "u")
    assert sha(b.f()) == str(g["f_sha256"])
    b.close()


@pytest.mark.parametrize("case", ["binary16_c1_s20", "binary16_c1_o3_s10", "binary16_c2_s20",
                                  "binary16_c2_o2_s10", "binary16_o4_g27_c1_s10"])
def test_binary_conserve_golden(golden, case):
    """cahn_hilliard_options_conserve 1 (compensated per-site update) and 2
    (global subtraction with the site-order sum), bit-exact against the
    reference run on one thread, through the staged kernels that the
    options select."""
    g = golden(case)
    n, nsteps, seed, order, a, b_, k, m, tau, phi0, amp = _binary_args(g)
    conserve = int(g["conserve"])
    print(f"case {case} conserve {conserve}", flush=True)
    stencil = int(g["stencil"]) if "stencil" in g else 7
    b = L.BinaryFluid((n, n, n), a=a, b=b_, kappa=k, mobility=m, order=order, tau=tau,
                      conserve=conserve, stencil=stencil)
    b.init_spinodal(seed, phi0, amp)
    b.step(nsteps)
    assert_exact(b.phi_field(), g["phi"], "phi")
    rho, u, _ = b.hydro_fields()
    assert_exact(rho, g["rho"], "rho")
    assert_exact(u, g["u"], "u")
    assert sha(b.f()) == str(g["f_sha256"])
    b.close()


@pytest.mark.parametrize("case", ["binary16_c2_s20", "binary16_c2_o2_s10"])
def test_conserve2_tree_sum_matches_golden(golden, case):
    """The default conserve-2 sum (compensated tree reduction) against the
    reference's one-thread run: the correction differs from the site-order
    one only by that sum's rounding, so every field stays within 1e-12
    relative (1e-12 absolute for u, whose values sit near zero)."""
    g = golden(case)
    n, nsteps, seed, order, a, b_, k, m, tau, phi0, amp = _binary_args(g)
    print(f"case {case} tree sum", flush=True)
    lib = L.lib()
    lib.ldw_conserve2_site_order(0)
    try:
        b = L.BinaryFluid((n, n, n), a=a, b=b_, kappa=k, mobility=m, order=order, tau=tau, conserve=2)
        b.init_spinodal(seed, phi0, amp)
        b.step(nsteps)
        phi = b.phi_field()
        rho, u, _ = b.hydro_fields()
        b.close()
    finally:
        lib.ldw_conserve2_site_order(1)
    assert np.max(np.abs(phi - g["phi"]) / np.maximum(np.abs(g["phi"]), 1e-3)) <= 1e-12
    assert np.max(np.abs(rho - g["rho"])) <= 1e-12
    assert np.max(np.abs(u - g["u"])) <= 1e-12


def test_conserve2_tree_sum_holds_the_sum_at_128():
    """At 128^3 the tree-sum mode keeps sum(phi) at its initial value to
    round-off over 50 steps, and it is far cheaper than the serial
    site-order sum (timed with HIP events on the library stream)."""
    import ctypes
    lib = L.lib()
    res = {}
    for mode in (0, 1):
        lib.ldw_conserve2_site_order(mode)
        try:
            b = L.BinaryFluid((128, 128, 128), tau=1.0, mobility=0.25, conserve=2)
            b.init_spinodal(8361235, 0.1, 0.1)
            _, p0 = b.conserved_sums()
            b.step(2)
            lib.ldw_stream_mark(0)
            b.step(20)
            lib.ldw_stream_mark(1)
            ms = ctypes.c_double()
            L._ck(lib.ldw_stream_elapsed(0, 1, ctypes.byref(ms)), "ldw_stream_elapsed")
            b.step(28)
            _, p1 = b.conserved_sums()
            b.close()
        finally:
            lib.ldw_conserve2_site_order(1)
        res[mode] = ms.value / 20
        assert abs(p1 - p0) <= 1e-10 * abs(p0), (mode, p0, p1)
    print(f"conserve 2 at 128^3: {res[0]:.3f} ms/step tree sum, {res[1]:.3f} ms/step site order")
    assert res[0] < 0.25 * res[1]


def test_conserve2_vs_oracle_nonuniform_box():
    """Conserve 2 on a box of odd sizes larger than one sum tile (2048
    sites), several steps, against the oracle bit for bit."""
    shape = (17, 13, 11)
    b = L.BinaryFluid(shape, a=-0.0625, b=0.0625, kappa=0.04, mobility=0.25, order=3, tau=0.9,
                      conserve=2)
    b.init_spinodal(4711, 0.2, 0.3)
    b.step(7)
    lb = O.lb_param(tau=0.9)
    fe = O.fe_param(a=-0.0625, b=0.0625, kappa=0.04, mobility=0.25, order=3, conserve=2)
    phi = O.spinodal(shape, 4711, 0.2, 0.3)
    f = O.equilibrium(shape, rho_uniform=1.0)
    f1, phi1, rho1, u1, _ = O.binary_steps_ext(shape, 7, lb, fe, f, phi,
                                               phi_init_sum=O.phi_init_sum(phi))
    assert_exact(b.phi_field(), phi1, "phi")
    assert_exact(b.f(), f1, "f")
    b.close()


@pytest.mark.parametrize("case", ["binary32_o1_s100", "binary32_o3_s200", "binary32_m045_s20"])
def test_binary32_long_golden(golden, case):
    g = golden(case)
    n, nsteps, seed, order, a, b_, k, m, tau, phi0, amp = _binary_args(g)
    b = L.BinaryFluid((n, n, n), a=a, b=b_, kappa=k, mobility=m, order=order, tau=tau)
    b.init_spinodal(seed, phi0, amp)
    b.step(nsteps)
    rho, u, _ = b.hydro_fields()
    for key, arr in (("phi", b.phi_field()), ("rho", rho), ("u", u), ("f", b.f())):
        assert sha(arr) == str(g[key + "_sha256"]), key
    b.close()


def test_single_fluid_c1_golden(golden):
    """C1: plain D3Q19 MRT, 32^3, tau 0.8, 100 steps; f, rho, u bit-exact."""
    g = golden("single32_s100")
    args = [str(a) for a in g["args"]]
    n, nsteps, seed, tau = int(args[1]), int(args[2]), int(args[3]), float(args[4])
    s = L.SingleFluid((n, n, n), tau=tau)
    s.init_random_velocity(seed)
    assert sha(s.f()) == str(g["f_init_sha256"])
    s.step(nsteps)
    rho, u, _ = s.hydro_fields()
    for key, arr in (("f", s.f()), ("rho", rho), ("u", u)):
        assert sha(arr) == str(g[key + "_sha256"]), key
    s.close()


@pytest.mark.parametrize("shape,order,nsteps,method,gm", [
    ((24, 20, 36), 1, 6, 0, (0.0, 0.0, 0.0)), ((16, 40, 12), 3, 4, 0, (0.0, 0.0, 0.0)),
    ((33, 17, 9), 2, 3, 0, (0.0, 0.0, 0.0)),
    ((21, 34, 70), 4, 5, 0, (0.0, 0.0, 0.0)),           # order 4, single-pass step, tile edges
    ((19, 23, 11), 5, 5, 1, (0.0, 0.0, 0.0)),           # order 5 wraps three sites on 11
    ((25, 12, 66), 4, 4, 1, (2e-4, -1e-4, 3e-4)),      # grad_mu with phi grad mu
    ((14, 30, 20), 2, 4, 0, (-3e-4, 0.0, 1e-4)),       # grad_mu, stress divergence
    ((128, 16, 64), 1, 4, 0, (0.0, 0.0, 0.0))])        # XCD-contiguous tile order (whole x-chunks per XCD)
def test_binary_nonuniform_box_vs_oracle(shape, order, nsteps, method, gm):
    """Non-cubic, odd sizes: the periodic wrap in every kernel, for every
    advection order and with an external chemical potential gradient."""
    print(f"case {shape} order={order} method={method} grad_mu={gm}", flush=True)
    fe = O.fe_param(order=order, mobility=0.25, force_method=method, grad_mu=gm)
    lb = O.lb_param(tau=0.9)
    phi0 = O.spinodal(shape, 99, 0.05, 0.1)
    f0 = O.equilibrium(shape, rho_uniform=1.0)
    f1, phi1, rho1, u1 = O.binary_steps(shape, nsteps, lb, fe, f0, phi0)
    b = L.BinaryFluid(shape, order=order, tau=0.9, mobility=0.25, grad_mu=gm,
                      force_method=L.FORCE_PHI_GRADMU if method else L.FORCE_STRESS_DIVERGENCE)
    b.init_spinodal(99, 0.05, 0.1)
    b.step(nsteps)
    assert_exact(b.phi_field(), phi1, "phi")
    rho, u, _ = b.hydro_fields()
    assert_exact(rho, rho1, "rho")
    assert_exact(u, u1, "u")
    assert_exact(b.f(), f1, "f")
    b.close()


NO_GM = (0.0, 0.0, 0.0)


@pytest.mark.parametrize("shape,conserve,precision,order,method,gm", [
    ((16, 16, 16), 0, 64, 1, 0, NO_GM),
    ((20, 16, 24), 1, 64, 2, 0, NO_GM),      # compensated update in the single-pass step
    ((20, 16, 24), 2, 64, 3, 0, NO_GM),      # global subtraction after the single-pass step
    ((20, 16, 24), 1, 32, 1, 0, NO_GM),
    ((20, 16, 24), 2, 32, 2, 0, NO_GM),
    ((20, 16, 24), 0, 64, 4, 0, NO_GM),      # order 4 in the single-pass step
    ((20, 16, 24), 1, 32, 4, 1, NO_GM),
    ((20, 16, 24), 0, 64, 5, 0, NO_GM),      # order 5: staged kernels either way
    ((20, 16, 24), 0, 64, 3, 1, (1e-3, 2e-3, -1e-3)),   # grad_mu with phi grad mu
    ((20, 16, 24), 1, 32, 2, 1, (1e-3, 2e-3, -1e-3)),
])
def test_staged_calls_equal_fused_step(shape, conserve, precision, order, method, gm):
    """The reference's call sequence through the C ABI equals ldw_step_binary,
    with cahn_hilliard_options_conserve 0, 1 and 2, FP64 and FP32, advection
    orders 1-5 and an external chemical potential gradient."""
    print(f"case staged vs fused {shape} conserve={conserve} fp{precision} order={order} "
          f"method={method} grad_mu={gm}", flush=True)
    kw = dict(tau=1.0, conserve=conserve, precision=precision, order=order, grad_mu=gm,
              force_method=L.FORCE_PHI_GRADMU if method else L.FORCE_STRESS_DIVERGENCE)
    nsteps = 3 if conserve == 0 else 6
    b1 = L.BinaryFluid(shape, **kw)
    b1.init_spinodal(5)
    b1.step(nsteps)
    b2 = L.BinaryFluid(shape, **kw)
    b2.init_spinodal(5)
    for _ in range(nsteps):
        b2.f_zero()
        b2.force_stage()
        b2.cahn_hilliard_stage()
        b2.u_zero()
        b2.collide(fe=b2.fe)
        b2.propagate()
    assert_exact(b2.phi_field(), b1.phi_field(), "phi")
    assert_exact(b2.f(), b1.f(), "f")
    r1, u1, F1 = b1.hydro_fields()      # force re-formed after the single-pass step
    r2, u2, F2 = b2.hydro_fields()
    assert_exact(r1, r2, "rho")
    assert_exact(u1, u2, "u")
    assert_exact(F1, F2, "force")
    b1.close()
    b2.close()


def test_stated_c2_mobility_blows_up_like_the_reference(golden):
    g = golden("binary32_m045_s40")
    n, nsteps, seed, order, a, b_, k, m, tau, phi0, amp = _binary_args(g)
    assert m == 0.45 and not bool(g["phi_finite"])
    b = L.BinaryFluid((n, n, n), a=a, b=b_, kappa=k, mobility=m, order=order, tau=tau)
    b.init_spinodal(seed, phi0, amp)
    b.step(nsteps)
    assert not np.isfinite(b.phi_field()).all()
    b.close()


def test_conservation_128_fp64():
    """C2 physics (M = 0.25) at 128^3: total density and phi conserved to
    round-off over 200 steps (compensated device sums)."""
    b = L.BinaryFluid((128, 128, 128), tau=1.0, mobility=0.25)
    b.init_spinodal(8361235)
    r0, p0 = b.conserved_sums()
    phi = b.phi_field()
    assert abs(p0 - __import__("math").fsum(phi)) <= 1e-12 * max(1.0, abs(p0))
    b.step(200)
    r1, p1 = b.conserved_sums()
    assert abs(r1 - r0) / r0 < 1e-13
    assert abs(p1 - p0) < 1e-10
    assert np.isfinite(b.phi_field()).all()
    b.close()


@pytest.mark.parametrize("order", [1, 3])
def test_binary_phi_gradmu_vs_oracle(order):
    """fe_force_method phi_gradmu through the fused force + Cahn-Hilliard pass."""
    shape = (20, 24, 16)
    fe = O.fe_param(order=order, mobility=0.25, force_method=1)
    lb = O.lb_param(tau=1.0)
    phi0 = O.spinodal(shape, 4321, 0.0, 0.1)
    f0 = O.equilibrium(shape, rho_uniform=1.0)
    f1, phi1, rho1, u1 = O.binary_steps(shape, 5, lb, fe, f0, phi0)
    b = L.BinaryFluid(shape, order=order, tau=1.0, mobility=0.25,
                      force_method=L.FORCE_PHI_GRADMU)
    b.init_spinodal(4321, 0.0, 0.1)
    b.step(5)
    assert_exact(b.phi_field(), phi1, "phi")
    rho, u, _ = b.hydro_fields()
    assert_exact(u, u1, "u")
    assert_exact(b.f(), f1, "f")
    b.close()


def test_fused_and_unfused_force_paths_agree():
    """phi_force_calculation followed by phi_cahn_hilliard runs the fused
    kernel; reading the force in between forces the separate kernels.  Both
    give the same bits."""
    shape = (32, 16, 24)
    b1 = L.BinaryFluid(shape, tau=1.0, order=3)
    b2 = L.BinaryFluid(shape, tau=1.0, order=3)
    for b in (b1, b2):
        b.init_spinodal(77, 0.0, 0.2)
        b.step(3)
    b1.f_zero(); b1.force_stage(); b1.cahn_hilliard_stage()          # fused
    b2.f_zero(); b2.force_stage(); _ = b2.hydro_fields(); b2.cahn_hilliard_stage()  # separate
    assert_exact(b1.phi_field(), b2.phi_field(), "phi")
    assert_exact(b1.hydro_fields()[2], b2.hydro_fields()[2], "force")
    b1.close()
    b2.close()


# The single-pass step's tiles and chunks: 16, 32 and 64 wide rows, one plane
# per block and several, columns and planes that the tile and the chunks cut
# unevenly, lattices smaller than a tile, too many columns for one round of
# blocks of either kernel (the first step is staged), and the large-lattice rule
# (rows of 32, chunks of 3 planes)
@pytest.mark.parametrize("shape", [(3, 5, 4), (7, 9, 15), (50, 17, 30), (12, 16, 33), (61, 40, 70), (3, 512, 340),
                                   (20, 203, 204)])
def test_step_tiles_match_oracle(shape):
    p = dict(a=-0.0625, b=0.0625, kappa=0.04, mobility=0.25)
    nsteps = 3
    print(f"step tiles {shape}", flush=True)
    b = L.BinaryFluid(shape, tau=1.0, fatal=True, **p)
    b.init_spinodal(77, 0.05, 0.1)
    b.step(nsteps)
    got = (b.f(), b.phi_field()) + b.hydro_fields()[:2]
    b.close()
    f0 = O.equilibrium(shape, rho_uniform=1.0)
    phi0 = O.spinodal(shape, 77, 0.05, 0.1)
    want = O.binary_steps(shape, nsteps, O.lb_param(tau=1.0), O.fe_param(**p), f0, phi0)
    for name, g, w in zip(("f", "phi", "rho", "u"), got, want):
        assert np.array_equal(g, w), name
