"""PIC element assembly on the GPU against the FP64 oracle on identical seeded swarms.

Bar: element matrices within 1e-12 (normwise per batch, FP64), G_e / f_e / approxS likewise,
per-particle viscosity within 1e-13 relative.
"""
import numpy as np
import pytest

from tests.helpers import OracleProblem, max_rel_err, rel_err, sinusoidal_temperature

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _system(dim, nel, ppc, seed, box=None):
    import earthbyte_underworld_amd as ust
    mn = (0.0,) * dim
    mx = box or (1.0,) * dim
    s = ust.StokesSystem(dim, nel, mn, mx)
    s.random_particle_layout(particlesPerCell=ppc, seed=seed)
    return s


def test_layout_matches_oracle(oracle):
    """RandomParticleLayout: MINSTD draws 3 per particle, cells in order (jump-ahead on the GPU)."""
    s = _system(2, (6, 5), 7, 13, box=(0.9142, 1.0))
    s.set_materials([__import__("earthbyte_underworld_amd").RheologyMaterial(
        [__import__("earthbyte_underworld_amd").MaterialViscosity(eta0=1.0)])])
    off, xi, w, _ = s.swarm()
    m = oracle.make_mesh(2, (6, 5), (0, 0), (0.9142, 1.0))
    coords = oracle.layout_random(m, 7, 13)
    xo, wo = oracle.map_particles(m, coords, off)
    assert np.array_equal(off, np.arange(0, 31) * 7)
    assert np.max(np.abs(xi[:, :2] - xo[:, :2])) < 1e-14
    assert np.array_equal(w, wo)


def test_layout_matches_oracle_3d(oracle):
    """The same in 3D (three draws per particle, x then y then z, cells in x-fastest order) on a non-cubic
    box with uneven counts."""
    import earthbyte_underworld_amd as ust
    nel, box = (4, 3, 5), (2.0, 1.0, 0.7)
    s = ust.StokesSystem(3, nel, (0.0, -1.0, 0.2), box)
    counts = np.random.default_rng(2).integers(1, 12, int(np.prod(nel)))
    s.random_particle_layout(seed=13, cell_counts=counts)
    off, xi, w, _ = s.swarm()
    m = oracle.make_mesh(3, nel, (0.0, -1.0, 0.2), box)
    coords = oracle.layout_random_counts(m, off, 13)  # the cells in order, each with its own count
    xo, wo = oracle.map_particles(m, coords, off)
    assert np.array_equal(np.diff(off), counts)
    assert np.max(np.abs(xi - xo)) < 1e-14
    assert np.array_equal(w, wo)


def test_layout_constant_weights_suite():
    """ConstantWeightsSuite.c:217-262 on the GPU layout: 1000 seeds of RandomParticleLayout (20 particles
    per cell, 2x2 elements on [0,4]^2) + ConstantWeights, element-0 integrals of the suite's six functions
    give the suite's error statistics.  The device's Lagrange weights integrate the quadratic-exact functions
    to the same values as the particle sum (detJ = 1 on these 2x2 elements)."""
    import earthbyte_underworld_amd as ust
    from tests import weights_suite as W
    s = ust.StokesSystem(2, W.NEL, W.BOX[0], W.BOX[1])
    s.set_materials([ust.RheologyMaterial([ust.MaterialViscosity(eta0=1.0)], density=0.0)])
    xs, ws = [], []
    lag = np.array([-1.0, 0.0, 1.0])
    qx, qy = lag[np.arange(9) % 3], lag[np.arange(9) // 3]
    for seed in range(W.SEEDS):
        s.random_particle_layout(particlesPerCell=W.PPC, seed=seed)
        off, xi, w, _ = s.swarm()
        xs.append(xi[:W.PPC])
        ws.append(w[:W.PPC])
        if seed < 50:
            s.assemble(gravity=0.0)
            WK = s.weights()[0][:, 0]
            for name in ("ConstantFunction", "LinearFunction", "QuadraticFunction"):
                f = W.FUNCTIONS[name][0]
                ref = float(np.sum(w[:W.PPC] * f(xi[:W.PPC, 0], xi[:W.PPC, 1])))
                assert abs(float(np.sum(WK * f(qx, qy))) - ref) < 1e-13 * max(1.0, abs(ref))
    stats = W.element_integrals(np.array(xs), np.array(ws), np.ones((W.SEEDS, W.PPC)))
    assert W.check(stats) == []


# particles per cell across the lane-segment widths of the assembly kernel (8, 12, 16, 21, 32, 64 and a
# count above 64 that loops)
@pytest.mark.parametrize("dim,nel,ppc", [(2, (8, 6), 20), (3, (5, 4, 3), 30), (3, (9, 5, 3), 3), (3, (9, 5, 3), 6),
                                         (2, (13, 7), 11), (3, (6, 5, 3), 16), (3, (6, 5, 3), 40),
                                         (2, (5, 4), 70)])
def test_element_matrices_isoviscous(oracle, dim, nel, ppc):
    import earthbyte_underworld_amd as ust
    s = _system(dim, nel, ppc, 13)
    s.set_materials([ust.RheologyMaterial([ust.MaterialViscosity(eta0=1.0)], density=1.0)])
    s.assemble(gravity=1.0)
    o = OracleProblem(s)
    assert max_rel_err(s.element_matrices(), o.Ke) < TOL
    assert max_rel_err(s.element_G(), o.Ge) < TOL
    assert max_rel_err(s.element_f(), o.fe) < TOL
    assert rel_err(s.approxS(), o.approxS) < TOL


@pytest.mark.parametrize("dim,nel,ppc", [(2, (16, 12), 20), (3, (6, 6, 4), 20)])
def test_element_matrices_multimaterial(oracle, dim, nel, ppc):
    """Spheres of log10 viscosity in [-2, 4] (the 3D viscosity-contrast case at a small size)."""
    import earthbyte_underworld_amd as ust
    s = _system(dim, nel, ppc, 7)
    rng = np.random.default_rng(3)
    mats = [ust.RheologyMaterial([ust.MaterialViscosity(eta0=1.0)], density=0.0)]
    shapes = []
    for k in range(6):
        mats.append(ust.RheologyMaterial([ust.MaterialViscosity(eta0=10 ** rng.uniform(-2, 4))], density=1.0))
        shapes.append(ust.Sphere(k + 1, rng.uniform(0.1, 0.9, dim), rng.uniform(0.1, 0.3)))
    s.set_materials(mats)
    s.assign_materials(shapes)
    s.assemble(gravity=1.0)
    o = OracleProblem(s)
    eta, _ = s.particle_viscosity()
    assert rel_err(eta, o.eta) < 1e-15
    assert max_rel_err(s.element_matrices(), o.Ke) < TOL
    assert max_rel_err(s.element_G(), o.Ge) < TOL
    assert max_rel_err(s.element_f(), o.fe) < TOL
    assert rel_err(s.approxS(), o.approxS) < TOL


def test_arrhenius_limiter_assembly(oracle):
    """Arrhenius with sinusoidal temperature, then ViscosityLimiter (testArrheniusWithLimiter.xml)."""
    import earthbyte_underworld_amd as ust
    s = _system(2, (10, 10), 25, 11)
    s.set_materials([ust.RheologyMaterial([ust.Arrhenius(eta0=1e-6, activationEnergy=27.63102112),
                                           ust.ViscosityLimiter(maxViscosity=10e4, minViscosity=10)])])
    T = sinusoidal_temperature(s)
    s.set_temperature(T)
    s.assemble()
    o = OracleProblem(s, temperature=T)
    eta, _ = s.particle_viscosity()
    assert rel_err(eta, o.eta) < 1e-14
    assert max_rel_err(s.element_matrices(), o.Ke) < TOL


def test_arrhenius_activation_volume_3d(oracle):
    import earthbyte_underworld_amd as ust
    s = _system(3, (4, 5, 3), 12, 5)
    s.set_materials([ust.RheologyMaterial([ust.Arrhenius(eta0=2.0, activationEnergy=3.0, activationVolume=1.5,
                                                         referenceTemperature=0.7)])])
    T = np.linspace(0.2, 1.0, s.nnodes)
    s.set_temperature(T)
    s.assemble()
    o = OracleProblem(s, temperature=T)
    eta, _ = s.particle_viscosity()
    assert rel_err(eta, o.eta) < 1e-14
    assert max_rel_err(s.element_matrices(), o.Ke) < TOL


@pytest.mark.parametrize("dim", [2, 3])
def test_yield_rheologies(oracle, dim):
    """Drucker-Prager and von Mises with a prescribed velocity and pressure (previous solution exists)."""
    import earthbyte_underworld_amd as ust
    nel = (12, 8) if dim == 2 else (6, 5, 4)
    s = _system(dim, nel, 16, 21)
    mats = [ust.RheologyMaterial([ust.Arrhenius(eta0=1.0, activationEnergy=5.0, referenceTemperature=1.0),
                                  ust.DruckerPrager(cohesion=0.3, frictionCoefficient=0.6, minimumViscosity=1e-2,
                                                    minimumYieldStress=0.05)]),
            ust.RheologyMaterial([ust.MaterialViscosity(eta0=3.0),
                                  ust.VonMises(cohesion=0.5, minimumViscosity=0.1)]),
            ust.RheologyMaterial([ust.MaterialViscosity(eta0=2.0),
                                  ust.VonMises(cohesion=0.4, minimumViscosity=0.1, strainRateSoftening=1)])]
    s.set_materials(mats)
    s.assign_materials([ust.Box(1, (0.0,) * dim, (0.5,) * dim), ust.Sphere(2, (0.7,) * dim, 0.2)])
    s.cohesion_noise(0.05, 99)
    rng = np.random.default_rng(1)
    u = 0.01 * rng.normal(size=s.ndof)
    p = rng.normal(size=s.nel)
    T = np.linspace(0.0, 1.0, s.nnodes)
    s.set_temperature(T)
    s.set_solution(u, p)
    s.set_previous_solution_exists(True)
    s.assemble()
    coh = s.cohesion_scale()
    assert np.all(np.abs(coh - 1.0) <= 0.05 + 1e-7) and coh.std() > 0.01
    o = OracleProblem(s, temperature=T, velocity=u, pressure=p, coh_scale=coh, prev=True)
    eta, yf = s.particle_viscosity()
    assert rel_err(eta, o.eta) < 1e-13
    assert np.array_equal(yf, o.yielded)
    assert 0.02 < yf.mean() < 0.98  # both branches exercised
    assert max_rel_err(s.element_matrices(), o.Ke) < TOL


def test_uneven_particle_counts(oracle):
    """Poisson-distributed counts clipped to [5, 60] (uneven batching across segment widths)."""
    import earthbyte_underworld_amd as ust
    s = ust.StokesSystem(2, (24, 12), (0, 0), (4.0, 1.0))
    counts = np.clip(np.random.default_rng(4).poisson(25, s.nel), 5, 60)
    counts[0], counts[1] = 5, 60
    s.random_particle_layout(seed=17, cell_counts=counts)
    s.set_materials([ust.RheologyMaterial([ust.MaterialViscosity(eta0=1.0)], density=1.0)])
    s.assemble()
    o = OracleProblem(s)
    assert np.array_equal(np.diff(o.off), counts)
    assert max_rel_err(s.element_matrices(), o.Ke) < TOL
    assert max_rel_err(s.element_f(), o.fe) < TOL


def test_plugin_callbacks_accumulate(oracle):
    """StiffnessMatrixTerm callbacks add (+=) their element block into elStiffMat."""
    import ctypes as C
    import earthbyte_underworld_amd as ust
    from earthbyte_underworld_amd import _lib as L
    s = _system(2, (4, 3), 10, 3)
    s.set_materials([ust.RheologyMaterial([ust.MaterialViscosity(eta0=2.0)], density=1.0)])
    s.assemble()
    lib = L.load()
    term_k, term_g = C.c_int(1), C.c_int(2)
    assert lib.ust_stg_bind_term(C.byref(term_k), s.ctx, L.TERM_CONSTITUTIVE) == 0
    assert lib.ust_stg_bind_term(C.byref(term_g), s.ctx, L.TERM_GRADIENT) == 0
    Ke = s.element_matrices()
    Ge = s.element_G()
    e = 7
    buf = np.full((8, 8), 1.0)
    rows = (C.POINTER(C.c_double) * 8)(*[buf[i].ctypes.data_as(C.POINTER(C.c_double)) for i in range(8)])
    lib.ust_ConstitutiveMatrixCartesian_AssembleElement(C.byref(term_k), None, e, None, None, rows)
    assert np.allclose(buf, 1.0 + Ke[e], rtol=0, atol=1e-14)
    gbuf = np.zeros((8, 1))
    grows = (C.POINTER(C.c_double) * 8)(*[gbuf[i].ctypes.data_as(C.POINTER(C.c_double)) for i in range(8)])
    lib.ust_GradientStiffnessMatrixTerm_AssembleElement(C.byref(term_g), None, e, None, None, grows)
    assert np.allclose(gbuf[:, 0], Ge[e], rtol=0, atol=1e-14)


def test_material_field_assignment():
    """ust_swarm_assign_materials_field: a nodal field interpolated at every particle by the Q1 shape functions
    of its element and binned to materials, against the same arithmetic in numpy on the downloaded swarm."""
    import earthbyte_underworld_amd as ust
    nel = (6, 5, 4)
    s = ust.StokesSystem(3, nel, (0.0, 0.0, 0.0), (2.0, 2.0, 1.0))
    s.random_particle_layout(particlesPerCell=9, seed=13)
    s.set_materials([ust.RheologyMaterial([ust.MaterialViscosity(eta0=10.0 ** (0.1 * k))]) for k in range(61)])
    f = np.random.default_rng(1).uniform(-3.5, 3.5, s.nnodes).astype(np.float32)
    corner = lambda i, j, k: [(i + a) + (nel[0] + 1) * ((j + b) + (nel[1] + 1) * (k + c))  # noqa: E731
                              for a in (0, 1) for b in (0, 1) for c in (0, 1)]
    f[corner(0, 0, 0)] = 10.0  # element 0 lies above the range, the last element below it
    f[corner(nel[0] - 1, nel[1] - 1, nel[2] - 1)] = -10.0
    s.assign_materials_field(f, -3.0, 3.0, 61)
    off, xi, _, mat = s.swarm()
    e = np.repeat(np.arange(s.nel), np.diff(off))
    ix, iy, iz = e % nel[0], (e // nel[0]) % nel[1], e // (nel[0] * nel[1])
    v = np.zeros(len(e))
    for a in range(8):
        b = [(a >> d) & 1 for d in range(3)]
        N = np.prod([0.5 * (1.0 + (2 * b[d] - 1) * xi[:, d]) for d in range(3)], axis=0)
        n = (ix + b[0]) + (nel[0] + 1) * ((iy + b[1]) + (nel[1] + 1) * (iz + b[2]))
        v += N * f[n].astype(np.float64)
    ref = np.clip(np.rint((v + 3.0) / 6.0 * 60.0), 0, 60).astype(np.uint8)
    assert np.array_equal(mat, ref)
    assert mat.min() == 0 and mat.max() == 60  # the clamp at both ends is exercised


def _oracle_buoyancy(b):
    o = __import__("oracle.oracle", fromlist=["Buoyancy"])
    ob = o.Buoyancy()
    import ctypes as C
    C.memmove(C.byref(ob), C.byref(b), C.sizeof(ob))
    return ob


@pytest.mark.parametrize("case", ["thermal_depth", "vertical_z", "direction", "adjust", "hydrostatic",
                                  "hydrostatic_moving", "thermal_2d"])
def test_buoyancy_force_term(oracle, case):
    """BuoyancyForceTerm.c:355-448 on the GPU against the oracle's density law and force: thermal (alpha, Tref)
    and compressible (beta, depthref) densities over a temperature field, VerticalAxis 2, gravityDirection,
    adjust, and a HydrostaticTerm background (still and with v, width, time), f_e within 1e-12."""
    import earthbyte_underworld_amd as ust
    dim = 2 if case == "thermal_2d" else 3
    nel = (7, 5) if dim == 2 else (5, 4, 3)
    box = (1.4, 1.0) if dim == 2 else (1.0, 0.8, 1.2)
    s = ust.StokesSystem(dim, nel, (0.0,) * dim, box)
    s.random_particle_layout(particlesPerCell=13, seed=5)
    mats = [ust.RheologyMaterial([ust.MaterialViscosity(eta0=1.0)], density=1.0, alpha=0.3,
                                 referenceTemperature=0.2, beta=0.5, referenceDepth=0.1),
            ust.RheologyMaterial([ust.MaterialViscosity(eta0=10.0)], density=-0.7, alpha=0.05,
                                 referenceTemperature=0.6)]
    s.set_materials(mats)
    s.assign_materials([ust.Everywhere(0), ust.Sphere(1, (0.5,) * dim, 0.3)])
    T = sinusoidal_temperature(s) + 0.1
    s.set_temperature(T)
    kw = {}
    if case == "vertical_z":
        kw = dict(VerticalAxis=2)
    elif case == "direction":
        kw = dict(gravityDirection=(0.36, -0.48, 0.8))
    elif case == "adjust":
        kw = dict(adjust=True)
    elif case == "hydrostatic":
        kw = dict(HydrostaticTerm=dict(upper_density=0.9, upper_alpha=0.1, lower_density=1.3, lower_alpha=0.02,
                                       height=0.7, material_boundary=0.35, T0=0.3, linear_coefficient=0.8,
                                       exponential_coefficient1=0.4, exponential_coefficient2=3.0))
    elif case == "hydrostatic_moving":
        kw = dict(HydrostaticTerm=dict(upper_density=0.9, upper_alpha=0.1, lower_density=1.3, lower_alpha=0.02,
                                       height=0.7, material_boundary=0.35, T0=0.3, linear_coefficient=0.8,
                                       v=0.5, width=2.0, time=0.6))
    b = ust.BuoyancyForceTerm(**kw)
    s.set_buoyancy(b)
    s.assemble(gravity=9.8)
    from tests.helpers import oracle_mesh, to_oracle_materials
    m = oracle_mesh(s)
    off, xi, w, mat = s.swarm()
    ob = _oracle_buoyancy(b)
    rho = oracle.eval_density(m, to_oracle_materials(s.materials), off, xi, mat.astype(np.int32), temperature=T,
                              buoyancy=ob)
    fe = oracle.element_forces(m, off, xi, w, rho, gravity=9.8, buoyancy=ob)
    assert np.max(np.abs(fe)) > 0.0
    assert max_rel_err(s.element_f(), fe) < TOL
    s.set_buoyancy(None)  # the defaults: VerticalAxis 1, no direction, no adjust, no background
    s.assemble(gravity=9.8)
    rho0 = oracle.eval_density(m, to_oracle_materials(s.materials), off, xi, mat.astype(np.int32), temperature=T)
    assert max_rel_err(s.element_f(), oracle.element_forces(m, off, xi, w, rho0, gravity=9.8)) < TOL


def _global_coords(s, off, xi):
    """Global particle coordinates from the cell-sorted local ones (rectilinear elements)."""
    ne = np.diff(off)
    e = np.repeat(np.arange(s.nel), ne)
    idx = [e % s.nel_axis[0], (e // s.nel_axis[0]) % s.nel_axis[1]]
    if s.dim == 3:
        idx.append(e // (s.nel_axis[0] * s.nel_axis[1]))
    x = np.zeros((len(e), 3))
    for d in range(s.dim):
        h = (s.max[d] - s.min[d]) / s.nel_axis[d]
        x[:, d] = s.min[d] + idx[d] * h + 0.5 * (xi[:, d] + 1.0) * h
    return x


@pytest.mark.parametrize("dim", [2, 3])
def test_strain_weakening_and_tensile_flag(oracle, dim):
    """StrainWeakening on DruckerPrager and VonMises (StrainWeakening.c:448-503, DruckerPrager.c:283-315,
    VonMises.c:194-199) against the oracle: viscosity, yield and tensile flags, the clamped weakening state and
    its increment per particle, and K_e; weakening values span unsoftened, partly and fully softened and
    negative (clamped) states, pressures both signs (tensile and compressive)."""
    import earthbyte_underworld_amd as ust
    from tests.helpers import oracle_mesh, to_oracle_materials
    nel = (12, 8) if dim == 2 else (6, 5, 4)
    s = _system(dim, nel, 16, 23)
    mats = [ust.RheologyMaterial([ust.MaterialViscosity(eta0=2.0),
                                  ust.DruckerPrager(cohesion=0.3, frictionCoefficient=0.6, minimumViscosity=1e-2,
                                                    minimumYieldStress=0.02, cohesionAfterSoftening=0.05,
                                                    frictionCoefficientAfterSoftening=0.2, StrainWeakening=1)]),
            ust.RheologyMaterial([ust.MaterialViscosity(eta0=3.0),
                                  ust.VonMises(cohesion=0.5, minimumViscosity=0.1, cohesionAfterSoftening=0.1,
                                               StrainWeakening=1)]),
            ust.RheologyMaterial([ust.MaterialViscosity(eta0=1.0),
                                  ust.DruckerPrager(cohesion=0.2, frictionCoefficient=0.3, minimumViscosity=1e-2)])]
    s.set_materials(mats)
    s.assign_materials([ust.Box(1, (0.0,) * dim, (0.5,) * dim), ust.Sphere(2, (0.7,) * dim, 0.2)])
    s.set_strain_weakening(ust.StrainWeakening(softeningStrain=0.8, healingRate=0.3))
    n = s.lib.ust_swarm_count(s.ctx)
    rng = np.random.default_rng(5)
    pfw = rng.uniform(-0.2, 1.2, n)
    s.set_strain_weakening_state(pfw, np.full(n, 9.0))
    u = 0.01 * rng.normal(size=s.ndof)
    p = rng.normal(size=s.nel)
    s.set_solution(u, p)
    s.set_previous_solution_exists(True)
    s.assemble()
    m = oracle_mesh(s)
    off, xi, w, mat = s.swarm()
    sw = {"pfw": pfw.copy(), "pfw_inc": np.full(n, 9.0), "softening_strain": 0.8, "healing_rate": 0.3}
    eta_o, y_o, t_o = oracle.eval_viscosity(m, to_oracle_materials(s.materials), off, xi, mat.astype(np.int32),
                                            velocity=u, pressure=p, previous_solution_exists=True,
                                            strain_weakening=sw, tensile=True)
    eta, y = s.particle_viscosity()
    pg, ig = s.strain_weakening()
    assert rel_err(eta, eta_o) < 1e-13
    assert np.array_equal(y, y_o) and 0.02 < y.mean() < 0.98  # both branches
    assert np.array_equal(s.tensile_failure(), t_o) and 0 < t_o.sum() < n
    assert np.array_equal(pg, sw["pfw"])
    assert (pg[mat != 2] >= 0).all() and np.array_equal(pg[mat == 2], pfw[mat == 2])  # clamped where read
    assert np.max(np.abs(ig - sw["pfw_inc"])) <= 1e-13 * np.max(np.abs(sw["pfw_inc"]))
    assert np.sum(ig == 9.0) == np.sum(mat == 2)  # the rheology without the flag assigns no increment
    Ke, _, _, _ = oracle.assemble_elements(m, off, xi, w, eta_o)
    assert max_rel_err(s.element_matrices(), Ke) < TOL
    # one time step of the weakening state, then the state follows its particles through an advection step
    s.strain_weakening_step(0.25)
    assert np.max(np.abs(s.strain_weakening()[0] - oracle.strain_weakening_step(sw["pfw"], sw["pfw_inc"], 0.25))) \
        < 1e-15
    x0 = _global_coords(s, off, xi)
    s.set_strain_weakening_state(x0[:, 0].copy(), np.zeros(n))
    vel = np.zeros(s.ndof)
    vel[0::dim] = 0.1
    s.set_solution(vel, p)
    s.advect(0.5, order=1, allowFallbackToFirstOrder=True)
    off2, xi2, _, _ = s.swarm()
    x1 = _global_coords(s, off2, xi2)
    pg, _ = s.strain_weakening()
    assert len(pg) == len(x1) < n
    assert np.max(np.abs(pg - (x1[:, 0] - 0.05))) < 1e-12


def test_strain_weakening_initial_damage(oracle):
    """_StrainWeakening_Initialise (StrainWeakening.c:318-399): the C library's srand(randomSeed)/rand() sequence
    drawn particle by particle in swarm order (one draw against initialDamageFraction, a second for the
    magnitude of a damaged particle), restricted to initialStrainShape and modulated by cos^2 / sin^2 of the
    wavenumber keys: restated here with the same C library calls; and the modulation pinned on its own: with
    every particle damaged the modulated state is the unmodulated one times cos^2(pi x k)."""
    import ctypes as C
    import earthbyte_underworld_amd as ust
    libc = C.CDLL(None)
    RAND_MAX = 2147483647
    s = _system(2, (8, 6), 12, 31)
    s.set_materials([ust.RheologyMaterial([ust.MaterialViscosity(eta0=1.0)])])
    off, xi, _, _ = s.swarm()
    x = _global_coords(s, off, xi)

    def reference(frac, factor, ss, seed, shape_box=None, cos_i=-1.0, sin_j=-1.0):
        libc.srand(C.c_uint(seed))
        out = np.zeros(len(x))
        for p in range(len(x)):
            v = 0.0
            if libc.rand() < RAND_MAX * frac:
                if shape_box is not None and not (shape_box[0] <= x[p, 0] <= shape_box[2]
                                                  and shape_box[1] <= x[p, 1] <= shape_box[3]):
                    continue
                v = factor * libc.rand() * ss / RAND_MAX
                if cos_i > 0:
                    v *= np.cos(np.pi * x[p, 0] * cos_i) ** 2
                if sin_j > 0:
                    v *= np.sin(np.pi * x[p, 1] * sin_j) ** 2
            out[p] = v
        return out

    cases = [dict(frac=0.3, factor=1.0, ss=0.5, seed=7), dict(frac=0.6, factor=2.0, ss=1.5, seed=0, cos_i=1.5),
             dict(frac=1.0, factor=1.0, ss=1.0, seed=3, shape_box=(0.2, 0.1, 0.7, 0.6), sin_j=2.0)]
    for c in cases:
        kw = dict(softeningStrain=c["ss"], initialDamageFraction=c["frac"], initialDamageFactor=c["factor"],
                  randomSeed=c["seed"], initialDamageWavenumberCosI=c.get("cos_i", -1.0),
                  initialDamageWavenumberSinJ=c.get("sin_j", -1.0))
        if "shape_box" in c:
            b = c["shape_box"]
            kw["initialStrainShape"] = ust.Box(0, (b[0], b[1], 0.0), (b[2], b[3], 1.0))
        s.set_strain_weakening(ust.StrainWeakening(**kw))
        s.strain_weakening_initialise()
        pfw, inc = s.strain_weakening()
        ref = reference(c["frac"], c["factor"], c["ss"], c["seed"], c.get("shape_box"), c.get("cos_i", -1.0),
                        c.get("sin_j", -1.0))
        assert np.max(np.abs(pfw - ref)) <= 1e-15 * max(1.0, ref.max()) and (inc == 0).all()
        assert 0 < np.count_nonzero(pfw) < len(pfw) or c["frac"] == 1.0
    s.set_strain_weakening(ust.StrainWeakening(softeningStrain=1.0, initialDamageFraction=1.0, randomSeed=4))
    s.strain_weakening_initialise()
    plain = s.strain_weakening()[0]
    s.set_strain_weakening(ust.StrainWeakening(softeningStrain=1.0, initialDamageFraction=1.0, randomSeed=4,
                                               initialDamageWavenumberCosI=0.75))
    s.strain_weakening_initialise()
    assert np.allclose(s.strain_weakening()[0], plain * np.cos(np.pi * x[:, 0] * 0.75) ** 2, rtol=1e-14, atol=0)


# counts at the edges of a matrix step (4 particles, 8 in 2D), of the 32 staged at a time and of the 64 loaded at a time
EDGE_COUNTS = [1, 3, 4, 5, 7, 8, 9, 31, 32, 33, 63, 64, 65, 1, 1, 130, 2, 96]


@pytest.mark.parametrize("dim,nel", [(2, (6, 3)), (3, (3, 3, 2)), (2, (18, 1)), (3, (1, 1, 18))])
def test_particle_weights_step_edges(oracle, dim, nel):
    import earthbyte_underworld_amd as ust
    s = ust.StokesSystem(dim, nel)
    s.random_particle_layout(seed=23, cell_counts=EDGE_COUNTS)
    s.set_materials([ust.RheologyMaterial([ust.MaterialViscosity(eta0=2.0)], density=1.5),
                     ust.RheologyMaterial([ust.MaterialViscosity(eta0=300.0),
                                           ust.ViscosityLimiter(maxViscosity=70.0, minViscosity=1.0)], density=0.5)])
    s.assign_materials([ust.Everywhere(0), ust.Box(1, (0.3,) * dim, (0.8,) * dim)])
    s.assemble()
    o = OracleProblem(s)
    eta, _ = s.particle_viscosity()
    assert rel_err(eta, o.eta) < 1e-13
    assert max_rel_err(s.element_matrices(), o.Ke) < TOL
    assert max_rel_err(s.element_G(), o.Ge) < TOL
    assert max_rel_err(s.element_f(), o.fe) < TOL


@pytest.mark.parametrize("dim,nel", [(2, (40, 3)), (3, (20, 3, 2)), (3, (64, 64, 33))])
def test_particle_weights_of_empty_elements(dim, nel):
    """Elements without particles get zero weights, at every place of a wave's 1 to 16 elements, and the others weights that
    add up to their particles'."""
    import earthbyte_underworld_amd as ust
    from tests.test_gpu_operators import _Dev
    rng = np.random.default_rng(3)
    ne = int(np.prod(nel))
    counts = rng.integers(0, 12, ne) * (rng.random(ne) < 0.6)
    counts[:3] = 0
    counts[-2:] = 0
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    xi = rng.uniform(-1, 1, (3, off[-1]))
    w = rng.uniform(0.1, 1.0, off[-1])
    s = ust.StokesSystem(dim, nel)
    s.set_materials([ust.RheologyMaterial([ust.MaterialViscosity(eta0=3.0)], density=2.0)])
    d = [_Dev(s.lib, a) for a in (off, xi[0], xi[1], xi[2], w)]
    assert s.lib.ust_swarm_upload_dev(s.ctx, int(off[-1]), *[a.p for a in d], None, None, int(counts.max())) == 0
    s.assemble()
    WK, WG, WF = s.weights()
    empty = counts == 0
    assert np.all(WK[:, empty] == 0) and np.all(WG[:, empty] == 0) and np.all(WF[:, empty] == 0)
    e = np.repeat(np.arange(ne), counts)
    detJ = float(np.prod([0.5 * (s.max[k] - s.min[k]) / nel[k] for k in range(dim)]))
    mass = np.bincount(e, weights=w * detJ, minlength=ne)
    # sums of the vertex and Lagrange functions are 1: each element's weights add to its particles' (5 roundings each)
    assert np.max(np.abs(WG.sum(0) - mass)) < 1e-14 * mass.max() * 5
    assert np.max(np.abs(WK.sum(0) - 3.0 * mass)) < 1e-14 * mass.max() * 50
    assert np.max(np.abs(WF.sum(0) - 2.0 * mass)) < 1e-14 * mass.max() * 10
    for a in d:
        a.free()


@pytest.mark.parametrize("dim,nel,ppc", [(3, (8, 8, 8), 100), (3, (8, 4, 4), 300), (2, (16, 16), 300)])
def test_rounding_of_the_particle_sums(dim, nel, ppc):
    """The sums' error does not grow with the particles.  Spacing, weights, viscosity and density are powers of two, so only
    the factors of a particle (independent: they average out) and the additions round.  A rounding's rms is about 0.4 u of
    the sum at that point (u = 2^-53); m additions in a chain of like terms come to 0.4 u sqrt(m / 3).  Blocks of 32
    particles, each of two chains of four steps: 0.4 u sqrt(8 / 3) = 0.65 u per block, independent between blocks, and the
    blocks' chain of at most 10: 0.75 u; together below 1 u.  One chain through all steps of four particles that round at
    each particle is 2.3 u at 100 and 4 u at 300.  Bar: 1.5 u in the 2-norm."""
    import earthbyte_underworld_amd as ust
    from tests.test_gpu_operators import _Dev
    rng = np.random.default_rng(11)
    ne = int(np.prod(nel))
    off = (np.arange(ne + 1) * ppc).astype(np.int32)
    xi = rng.uniform(-1, 1, (3, off[-1]))
    w = np.full(off[-1], 2.0 ** -6)
    s = ust.StokesSystem(dim, nel)
    s.set_materials([ust.RheologyMaterial([ust.MaterialViscosity(eta0=4.0)], density=2.0)])
    d = [_Dev(s.lib, a) for a in (off, xi[0], xi[1], xi[2], w)]
    assert s.lib.ust_swarm_upload_dev(s.ctx, int(off[-1]), *[a.p for a in d], None, None, ppc) == 0
    s.assemble()
    got = s.weights()
    X = xi[:dim].astype(np.longdouble)
    detJ = float(np.prod([0.5 / k for k in nel]))
    lag = [(x * (x - 1) / 2, 1 - x * x, x * (x + 1) / 2) for x in X]
    lin = [((1 - x) / 2, (1 + x) / 2) for x in X]

    def sums(factors, base, scale):
        rows = []
        for q in range(base ** dim):
            v = np.full(off[-1], scale, np.longdouble)
            for k in range(dim):
                v = v * factors[k][(q // base ** k) % base]
            rows.append(np.add.reduceat(v, off[:-1]))
        return np.array(rows)

    one = detJ * 2.0 ** -6
    for name, g, r in zip(("WK", "WG", "WF"), got,
                          (sums(lag, 3, 4.0 * one), sums(lin, 2, one), sums(lin, 2, 2.0 * one))):
        err = float(np.sqrt(np.sum((g.astype(np.longdouble) - r) ** 2) / np.sum(r ** 2)))
        assert err < 1.5 * 2.0 ** -53, (name, err * 2.0 ** 53)
    for a in d:
        a.free()


# fewer elements than a block, partial blocks, and more than the passes' blocks take at once (1024 x 256)
@pytest.mark.parametrize("dim,nel", [(2, (5, 3)), (2, (600, 500)), (3, (3, 2, 5)), (3, (70, 65, 60))])
def test_derived_terms_of_an_assembly(dim, nel):
    """ust_k_derive on random weights and masks: approxS as ust_k_uzawa_diag (the same device code: bit-equal), h = 0, and
    f, ||G 1||^2 and the largest row sum of |G^T| against NumPy sums (up to a few hundred roundings: 1e-13)."""
    import ctypes as C
    import earthbyte_underworld_amd as ust  # noqa: F401  (loads the library)
    from earthbyte_underworld_amd import _lib as L
    from tests.test_gpu_operators import _Dev, _grid
    lib = L.load()
    g = _grid(dim, nel)
    ne, nv = int(np.prod(nel)), 1 << dim
    nn = [k + 1 for k in nel]
    n = int(np.prod(nn))
    rng = np.random.default_rng(8)
    wl = lib.ust_k_weights_len(C.byref(g))
    WG, WF = rng.uniform(0.5, 1.0, (nv, ne)), rng.normal(size=(nv, ne))
    mask = (rng.random((n, dim)) < 0.2).astype(np.uint8)
    dirn = np.array([0.0, -1.0, 0.3])
    dW, dG, dF = _Dev(lib, rng.uniform(0.1, 1.0, wl)), _Dev(lib, WG), _Dev(lib, WF)
    dm, da, da2 = _Dev(lib, mask), _Dev(lib, np.full(ne, np.nan)), _Dev(lib, np.zeros(ne))
    df, dh = _Dev(lib, np.full(n * dim, np.nan)), _Dev(lib, np.full(ne, np.nan))
    dp, dn = _Dev(lib, np.zeros(2048)), _Dev(lib, np.zeros(2))
    assert lib.ust_k_derive(C.byref(g), dW.p, dG.p, dF.p, 2.5, dirn.ctypes.data_as(C.c_void_p), dm.p, da.p, df.p, dh.p,
                            dp.p, dn.p, None) == 0
    assert lib.ust_k_uzawa_diag(C.byref(g), dW.p, dG.p, da2.p, None) == 0
    assert np.array_equal(da.get(), da2.get()) and np.all(dh.get() == 0.0)
    e = np.arange(ne)
    ijk = [e % nel[0], (e // nel[0]) % nel[1]] + ([e // (nel[0] * nel[1])] if dim == 3 else [])
    f, g1, rows = np.zeros((n, dim)), np.zeros((n, dim)), np.zeros(ne)
    for a in range(nv):
        node = np.zeros(ne, np.int64)
        for k in reversed(range(dim)):
            node = node * nn[k] + ijk[k] + ((a >> k) & 1)
        for i in range(dim):
            Ge = -(2 * ((a >> i) & 1) - 1) / g.h[i] * (WG[a] + WG[a ^ (1 << i)])
            np.add.at(g1[:, i], node, Ge)
            rows += np.where(mask[node, i], 0.0, np.abs(Ge))
            np.add.at(f[:, i], node, 2.5 * dirn[i] * WF[a])
    f[mask != 0] = 0.0
    norms = dn.get()
    assert rel_err(df.get(), f.reshape(-1)) < 1e-13
    assert abs(norms[0] - np.sum(g1[mask == 0] ** 2)) < 1e-13 * norms[0]
    assert abs(norms[1] - rows.max()) < 1e-14 * norms[1]
    for x in (dW, dG, dF, dm, da, da2, df, dh, dp, dn):
        x.free()
