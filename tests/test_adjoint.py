"""Tangent and adjoint of the level-1 residual on the GPU.

The reference has no differentiated code, so these are pinned by the
mathematics: the tangent against central finite differences of the
residual the library itself computes (FLITE_OP_RHS, parity-checked against
the oracle elsewhere), the adjoint against the tangent by the dot-product
identity <lam, J du> = <J^T lam, du>, and the drag gradient against finite
differences of the drag.  Euler, first-order HLLC, M=0.8, alpha=1.25 deg
(the discrete-adjoint case's conditions) on a jittered 8^3 bump box and a
12^3 one after a few cycles, so that every flux branch and both boundary
kinds (wall and farfield) are exercised.
"""
import numpy as np
import pytest
import torch  # torch before the first context: its device init after one has failed on this image

from flite3d_amd.device import Solver
from oracle import Oracle

from cases import euler, levels

pytestmark = pytest.mark.gpu

H = 1e-7


def make(n, cycles, order=1):
    lv = levels(n, 2, jitter=0.15)
    iv = euler(order, machnumber=0.8, alpha=1.25, cflnumber=2.0)
    s = Solver(iv.to_struct(), list(lv))
    s.init_freestream()
    for c in range(1, cycles + 1):
        s.cycle(c)
    return s, lv


def residual(s, u):
    s.set(1, "U", u)
    s.apply(1, "PRESSURE")
    s.apply(1, "RHS")
    return s.get(1, "RHS")[:5]


def directions(rng, u, k):
    """Unit-norm random perturbations, scaled per component to the state."""
    out = []
    for _ in range(k):
        d = rng.standard_normal((5, u.shape[1])) * np.abs(u[:5]).max(axis=1, keepdims=True)
        out.append(d / np.linalg.norm(d))
    return out


@pytest.mark.parametrize("n,cycles", [(8, 0), (12, 5)])
def test_tangent_matches_central_differences(n, cycles):
    print(f"[case] tangent FD n={n} cycles={cycles}", flush=True)
    s, lv = make(n, cycles)
    o = oracle_for(s, lv)  # central differences of the oracle's residual
    u = s.get(1, "U")
    rng = np.random.default_rng(1)
    for du in directions(rng, u, 4):
        jt = s.tangent(du)
        up, um = u.copy(), u.copy()
        up[:5] += H * du
        um[:5] -= H * du
        fd = (residual(o, up) - residual(o, um)) / (2 * H)
        err = np.abs(fd - jt).max() / np.abs(jt).max()
        assert err < 1e-5, err
    s.close()
    o.close()


@pytest.mark.parametrize("n,cycles", [(8, 0), (12, 5)])
def test_adjoint_dot_product(n, cycles):
    print(f"[case] adjoint dot product n={n} cycles={cycles}", flush=True)
    s, lv = make(n, cycles)
    u = s.get(1, "U")
    rng = np.random.default_rng(2)
    for du, lam in zip(directions(rng, u, 4), directions(rng, u, 4)):
        a = np.sum(lam * s.tangent(du))
        b = np.sum(s.adjoint(lam) * du)
        assert abs(a - b) <= 1e-12 * max(abs(a), abs(b)) + 1e-300, (a, b)
    s.close()


def test_adjoint_columns_are_jacobian_rows():
    """J^T e_k for unit vectors e_k equals row k of J built column by
    column from the tangent (small mesh, a few nodes)."""
    print("[case] adjoint vs explicit Jacobian rows", flush=True)
    s, lv = make(8, 2)
    u = s.get(1, "U")
    n = u.shape[1]
    rng = np.random.default_rng(3)
    for node in rng.choice(n, 3, replace=False):
        for comp in (0, 4):
            e = np.zeros((5, n))
            e[comp, node] = 1.0
            row = s.adjoint(e)  # J^T e = row (node, comp) of J
            for j in rng.choice(n, 4, replace=False):
                for c in range(5):
                    d = np.zeros((5, n))
                    d[c, j] = 1.0
                    assert abs(s.tangent(d)[comp, node] - row[c, j]) <= 1e-12 * (1 + abs(row[c, j]))
    s.close()


def test_drag_gradient_matches_central_differences():
    print("[case] drag gradient FD", flush=True)
    s, lv = make(12, 5)
    u = s.get(1, "U")
    drag0, g = s.drag_gradient()
    assert np.isfinite(drag0) and np.abs(g).max() > 0
    rng = np.random.default_rng(4)
    for du in directions(rng, u, 4):
        up, um = u.copy(), u.copy()
        up[:5] += H * du
        um[:5] -= H * du
        s.set(1, "U", up)
        dp, _ = s.drag_gradient()
        s.set(1, "U", um)
        dm, _ = s.drag_gradient()
        fd = (dp - dm) / (2 * H)
        an = np.sum(g * du)
        assert abs(fd - an) <= 1e-6 * max(abs(an), 1e-12), (fd, an)
    s.set(1, "U", u)
    s.close()


# Second order (MUSCL reconstruction with LED clipping): the residual is
# piecewise smooth, with kinks where a limiter switch flips (the minmod
# choice, the clip to the side half-length, the neighbour that sets a
# bound) or where a Roe eigenvalue |u.n| crosses zero.  A state a few
# cycles from freestream is nearly uniform away from the bump, so equal
# neighbour values put bound switches right at the state; the
# linearisation is therefore checked about a smooth non-uniform state with
# no equal neighbour values and no zero velocity component.
def smooth_state(lv, u):
    x, y, z = lv[0].coords
    f = [np.sin(2.1 * x + 0.4 * z + 0.31) * np.cos(1.7 * y + 0.23),
         np.cos(1.3 * x - 0.5 * z + 0.8 * y + 0.17),
         np.sin(1.9 * y + z - 0.3 * x + 0.57),
         np.cos(2.3 * z + 0.7 * x + 0.2 * y + 0.41),
         np.sin(1.1 * x + 1.4 * y - 0.6 * z + 0.73)]
    out = u.copy()
    for c in range(5):
        out[c] = u[c] * (1 + 0.05 * f[c]) + (0.02 * (1.5 + f[c]) if c in (2, 3) else 0.0)
    return out


def make_smooth(n, order):
    lv = levels(n, 2, jitter=0.15)
    s = Solver(euler(order, machnumber=0.8, alpha=1.25, cflnumber=2.0).to_struct(), list(lv))
    s.init_freestream()
    u = smooth_state(lv, s.get(1, "U"))
    s.set(1, "U", u)
    s.apply(1, "PRESSURE")
    return s, lv, u


@pytest.mark.parametrize("n", [8, 12])
def test_second_order_tangent_matches_finite_differences(n):
    """Every entry of J du equals the central difference, or, where a
    switch lies within H of the state (the residual is only piecewise
    smooth), the one-sided difference taken on the state's side of it;
    such entries are rare."""
    print(f"[case] second-order tangent FD n={n}", flush=True)
    s, lv, u = make_smooth(n, 2)
    o = oracle_for(s, lv)  # differences of the oracle's residual
    rng = np.random.default_rng(5)
    one_sided = 0
    for du in directions(rng, u, 4):
        jt = s.tangent(du)
        r0 = residual(o, u)
        up, um = u.copy(), u.copy()
        up[:5] += H * du
        um[:5] -= H * du
        rp, rm = residual(o, up), residual(o, um)
        tol = 1e-6 * np.abs(jt).max()
        central = np.abs((rp - rm) / (2 * H) - jt) <= tol
        fwd = np.abs((rp - r0) / H - jt) <= tol
        bwd = np.abs((r0 - rm) / H - jt) <= tol
        assert np.all(central | fwd | bwd), np.argwhere(~(central | fwd | bwd))[:5]
        one_sided += int((~central).sum())
    assert one_sided <= 0.001 * jt.size * 4, one_sided
    s.close()
    o.close()


def test_second_order_tangent_differs_from_first_order():
    """The reconstruction's derivatives contribute: on the same state the
    second-order Jacobian is not the first-order one, and the LED clipping
    changes it again."""
    print("[case] second- vs first-order tangent", flush=True)
    s2, lv, u = make_smooth(8, 2)
    du = directions(np.random.default_rng(6), u, 1)[0]
    j2 = s2.tangent(du)
    s2.close()
    for kw in (dict(hllcfluxorder=1), dict(automaticlipping=0)):
        args = dict(machnumber=0.8, alpha=1.25, cflnumber=2.0)
        args.update(kw)
        s = Solver(euler(2, **args).to_struct(), list(lv))
        s.set(1, "U", u)
        s.init_from_state()
        j = s.tangent(du)
        s.close()
        assert np.abs(j2 - j).max() > 1e-3 * np.abs(j2).max(), kw


@pytest.mark.parametrize("n,smooth", [(8, True), (12, True), (12, False)])
def test_second_order_adjoint_dot_product(n, smooth):
    """<lam, J du> = <J^T lam, du>; the identity holds at any state, also
    one with limiter switches at the state (a few cycles from freestream)."""
    print(f"[case] second-order adjoint dot product n={n} smooth={smooth}", flush=True)
    if smooth:
        s, lv, u = make_smooth(n, 2)
    else:
        s, lv = make(n, 5, order=2)
        u = s.get(1, "U")
    rng = np.random.default_rng(7)
    for du, lam in zip(directions(rng, u, 4), directions(rng, u, 4)):
        a = np.sum(lam * s.tangent(du))
        b = np.sum(s.adjoint(lam) * du)
        assert abs(a - b) <= 1e-12 * max(abs(a), abs(b)) + 1e-300, (a, b)
    s.close()


def test_second_order_adjoint_columns_are_jacobian_rows():
    """J^T e_k equals row k of J, over the nodes of k's two-ring (the
    second-order stencil: the neighbours' gradients and bounds)."""
    print("[case] second-order adjoint vs explicit Jacobian rows", flush=True)
    s, lv, u = make_smooth(8, 2)
    n = u.shape[1]
    ea, eb = lv[0].side_index
    nbr = [set() for _ in range(n)]
    for a, b in zip(ea, eb):
        nbr[a].add(b)
        nbr[b].add(a)
    rng = np.random.default_rng(8)
    for node in rng.choice(n, 2, replace=False):
        ring = set(nbr[node])
        for m in list(ring):
            ring |= nbr[m]
        cols = rng.choice(sorted(ring), 6, replace=False)
        for comp in (0, 1, 4):
            e = np.zeros((5, n))
            e[comp, node] = 1.0
            row = s.adjoint(e)
            for j in cols:
                for c in range(5):
                    d = np.zeros((5, n))
                    d[c, j] = 1.0
                    t = s.tangent(d)[comp, node]
                    assert abs(t - row[c, j]) <= 1e-12 * (1 + abs(row[c, j])), (node, comp, j, c, t, row[c, j])
        # the row reaches the second ring
        far = sorted(j for j in ring if j not in nbr[node] and j != node)
        e = np.zeros((5, n))
        e[1, node] = 1.0
        assert np.abs(s.adjoint(e)[:, far]).max() > 0
    s.close()


@pytest.mark.parametrize("order", [1, 2])
def test_first_apply_on_a_fresh_context_equals_the_second(order):
    """The scratch of the tangent and adjoint is allocated (and zeroed) on
    the first call: that call's result must equal a repeat's."""
    print(f"[case] fresh-context tangent/adjoint order={order}", flush=True)
    for k in range(2):
        s, lv, u = make_smooth(12, order)
        rng = np.random.default_rng(9 + k)
        du, lam = directions(rng, u, 2)
        if k == 0:
            a1, t1 = s.adjoint(lam), s.tangent(du)
            a2, t2 = s.adjoint(lam), s.tangent(du)
        else:
            t1, a1 = s.tangent(du), s.adjoint(lam)
            t2, a2 = s.tangent(du), s.adjoint(lam)
        assert np.array_equal(a1, a2) and np.array_equal(t1, t2)
        s.close()


# ---- laminar flow: the viscous term linearised too ----
def make_laminar(n, order):
    """The smooth state on the freestream before the no-slip condition (the
    wall nodes' zero velocity would tie neighbouring values)."""
    from cases import laminar
    lv = levels(n, 2, jitter=0.15)
    iv = laminar(hllcfluxorder=order, reynoldsnumber=200.0, wallsareisentropic=True)
    s = Solver(iv.to_struct(), list(lv))
    s.init_freestream()
    inf = np.array(iv.inflowfield[0])
    base = np.zeros((6, lv[0].n_nodes))
    base[:5] = inf[:5, None]
    base[1:4] *= inf[0]
    base[5] = s.get(1, "U")[5]
    u = smooth_state(lv, base)
    s.set(1, "U", u)
    s.apply(1, "PRESSURE")
    return s, lv, u


def oracle_for(s, lv):
    """The oracle on the solver's fine level and parameters: the finite
    differences below are of its residual, the CPU restatement of the
    reference's, not of the GPU's."""
    o = Oracle(s.params[0], [lv[0]])
    o.init_freestream()
    return o


def viscous_alone(s):
    """The viscous op on a cleared dissipation array: makeViscosityTerm
    subtracts into dissipation(:,2:5) (the oracle keeps what is there)."""
    s.set(1, "DISSIPATION", np.zeros((5, s.n(1))))
    s.apply(1, "VISCOUS")


def residual_laminar(s, u):
    """makeRHS plus the viscous dissipation (dissipation(:,2:5) = -viscous)."""
    s.set(1, "U", u)
    s.apply(1, "PRESSURE")
    s.apply(1, "RHS")
    viscous_alone(s)
    return s.get(1, "RHS")[:5] + s.get(1, "DISSIPATION")[:5]


@pytest.mark.parametrize("order", [1, 2])
def test_laminar_tangent_matches_finite_differences(order):
    """Every entry equals the central difference of the oracle's residual,
    or, at second order, a one-sided one where a limiter switch lies within
    H; the viscous part
    (Green-Gauss gradients of u, v, w, T, Sutherland viscosity, adiabatic
    wall projection, edge and boundary fluxes) is smooth."""
    print(f"[case] laminar tangent FD order={order}", flush=True)
    s, lv, u = make_laminar(8, order)
    o = oracle_for(s, lv)
    rng = np.random.default_rng(31)
    one_sided = 0
    for du in directions(rng, u, 3):
        jt = s.tangent(du)
        r0 = residual_laminar(o, u)
        up, um = u.copy(), u.copy()
        up[:5] += H * du
        um[:5] -= H * du
        rp, rm = residual_laminar(o, up), residual_laminar(o, um)
        tol = 1e-6 * np.abs(jt).max()
        central = np.abs((rp - rm) / (2 * H) - jt) <= tol
        fwd = np.abs((rp - r0) / H - jt) <= tol
        bwd = np.abs((r0 - rm) / H - jt) <= tol
        ok = central | fwd | bwd if order == 2 else central
        assert np.all(ok), (np.argwhere(~ok)[:5], np.abs((rp - rm) / (2 * H) - jt).max() / np.abs(jt).max())
        one_sided += int((~central).sum())
    assert one_sided <= 0.001 * jt.size * 3, one_sided
    # the viscous part is really there: the inviscid Jacobian differs
    from cases import euler as _euler
    si = Solver(_euler(order).to_struct(), list(lv))
    si.set(1, "U", u)
    si.init_from_state()
    du = directions(rng, u, 1)[0]
    assert np.abs(s.tangent(du) - si.tangent(du)).max() > 1e-2 * np.abs(s.tangent(du)).max()
    si.close()
    s.close()
    o.close()


@pytest.mark.parametrize("order", [1, 2])
def test_laminar_adjoint_dot_product(order):
    print(f"[case] laminar adjoint dot product order={order}", flush=True)
    s, lv, u = make_laminar(8, order)
    rng = np.random.default_rng(32)
    for du, lam in zip(directions(rng, u, 4), directions(rng, u, 4)):
        a = np.sum(lam * s.tangent(du))
        b = np.sum(s.adjoint(lam) * du)
        assert abs(a - b) <= 1e-12 * max(abs(a), abs(b)) + 1e-300, (a, b)
    s.close()


def test_linearisation_rejects_unsupported_settings():
    """Spalart-Allmaras runs in the tangent, the adjoint, the drag's state
    gradient and the mesh adjoint (6 components); the first-order inviscid
    entry points (metric adjoint, drag metric gradient) refuse it."""
    from flite3d_amd.device import DeviceError
    from cases import rans
    lv = levels(8, 2, first_cell=0.005)
    s = Solver(rans().to_struct(), list(lv))
    s.init_freestream()
    n = lv[0].n_nodes
    assert s.tangent(np.zeros((6, n))).shape == (6, n)
    assert s.adjoint(np.zeros((6, n))).shape == (6, n)
    assert s.drag_gradient()[1].shape == (6, n)
    assert s.mesh_adjoint(np.zeros((6, n)))[4].shape == (n,)
    with pytest.raises(DeviceError):
        s.metric_adjoint(np.zeros((5, n)))
    with pytest.raises(DeviceError):
        s.drag_metric_gradient()
    s.close()


# ---- RANS-SA: the Spalart-Allmaras terms in the tangent ----
def make_rans(n, order, re=1.0e4):
    """A smooth state with nu~ of a few times the laminar viscosity (chi of
    a few units, where the eddy viscosity, the source's fv1/fv2/fw and the
    diffusion all vary), on the freestream before the wall conditions."""
    from cases import rans
    lv = levels(n, 2, jitter=0.15)
    iv = rans(hllcfluxorder=order, reynoldsnumber=re)
    s = Solver(iv.to_struct(), list(lv))
    s.init_freestream()
    inf = np.array(iv.inflowfield[0])
    base = np.zeros((6, lv[0].n_nodes))
    base[:5] = inf[:5, None]
    base[1:4] *= inf[0]
    u = smooth_state(lv, base)
    x, y, z = lv[0].coords
    u[5] = 3.0 * (1.0 + 0.3 * np.sin(1.7 * x + 0.9 * y - 1.3 * z + 0.2))
    s.set(1, "U", u)
    s.apply(1, "PRESSURE")
    return s, lv, u


def residual_rans(s, u):
    """The RANS-SA residual the tangent linearises: makeRHS and the SA
    convection and source (RHS), plus the viscous dissipation (VISCOUS, with
    the eddy viscosity) on the mean flow and the SA diffusion (SA_DIFFUSION)
    on nu~."""
    s.set(1, "U", u)
    s.apply(1, "PRESSURE")
    viscous_alone(s)
    s.apply(1, "SA_DIFFUSION")
    s.apply(1, "RHS")
    r = s.get(1, "RHS")[:6].copy()
    r[:5] += s.get(1, "DISSIPATION")[:5]
    r[5] += s.get(1, "TURB_DIFFUSION")[0]
    return r


def directions6(rng, u, k):
    out = []
    for _ in range(k):
        d = rng.standard_normal((6, u.shape[1])) * np.abs(u[:6]).max(axis=1, keepdims=True)
        out.append(d / np.linalg.norm(d))
    return out


@pytest.mark.parametrize("order", [1, 2])
def test_rans_tangent_matches_finite_differences(order):
    """Every entry of the 6-component tangent equals the central difference
    of the oracle's RANS-SA residual, or a one-sided one where a switch
    (limiter, the source's clips) lies within H."""
    print(f"[case] RANS-SA tangent FD order={order}", flush=True)
    s, lv, u = make_rans(8, order)
    o = oracle_for(s, lv)
    rng = np.random.default_rng(41)
    one_sided = 0
    for du in directions6(rng, u, 3):
        jt = s.tangent(du)
        assert jt.shape == (6, lv[0].n_nodes)
        r0 = residual_rans(o, u)
        up, um = u.copy(), u.copy()
        up[:6] += H * du
        um[:6] -= H * du
        rp, rm = residual_rans(o, up), residual_rans(o, um)
        for c in range(6):  # each component on its own scale (nu~'s residual is small)
            tol = 1e-6 * np.abs(jt[c]).max() + 1e-300
            central = np.abs((rp[c] - rm[c]) / (2 * H) - jt[c]) <= tol
            fwd = np.abs((rp[c] - r0[c]) / H - jt[c]) <= tol
            bwd = np.abs((r0[c] - rm[c]) / H - jt[c]) <= tol
            ok = central | fwd | bwd
            assert np.all(ok), (c, np.argwhere(~ok)[:5],
                                np.abs((rp[c] - rm[c]) / (2 * H) - jt[c]).max() / np.abs(jt[c]).max())
            one_sided += int((~central).sum())
    assert one_sided <= 0.002 * jt.size * 3, one_sided
    s.close()
    o.close()


def test_rans_tangent_couples_nu_and_mean_flow():
    """A nu~-only direction moves the mean flow's residual (eddy viscosity
    in the stress) and nu~'s (convection, diffusion, source); a mean-flow
    direction moves nu~'s residual (convection velocity, vorticity,
    laminar viscosity)."""
    print("[case] RANS-SA tangent coupling", flush=True)
    s, lv, u = make_rans(8, 1)
    rng = np.random.default_rng(43)
    dn = np.zeros((6, lv[0].n_nodes))
    dn[5] = rng.standard_normal(lv[0].n_nodes)
    jn = s.tangent(dn)
    assert np.abs(jn[1:5]).max() > 0 and np.abs(jn[5]).max() > 0
    dm = np.zeros((6, lv[0].n_nodes))
    dm[1:4] = rng.standard_normal((3, lv[0].n_nodes)) * np.abs(u[1:4]).max()
    jm = s.tangent(dm)
    assert np.abs(jm[5]).max() > 0
    s.close()


@pytest.mark.parametrize("order", [1, 2])
def test_rans_adjoint_dot_product(order):
    """<lam, J du> = <J^T lam, du> for the RANS-SA residual, over the whole
    vectors and over blocks that isolate the couplings: nu~'s row against
    each state component (convection, diffusion and source) and the mean
    flow's rows against nu~ (the eddy viscosity)."""
    print(f"[case] RANS-SA adjoint dot product order={order}", flush=True)
    s, lv, u = make_rans(8, order)
    rng = np.random.default_rng(47)
    blocks = [(range(6), range(6)), ([5], range(6)), ([5], [0]), ([5], [1, 2, 3]), ([5], [4]), ([5], [5]),
              ([1, 2, 3, 4], [5]), (range(5), range(5))]
    for rows, cols in blocks:
        du, lam = directions6(rng, u, 2)
        du[[c for c in range(6) if c not in cols]] = 0.0
        lam[[c for c in range(6) if c not in rows]] = 0.0
        a = np.sum(lam * s.tangent(du))
        b = np.sum(s.adjoint(lam) * du)
        assert abs(a) > 0, (rows, cols)
        assert abs(a - b) <= 1e-12 * max(abs(a), abs(b)), (list(rows), list(cols), a, b)
    s.close()


def test_rans_adjoint_columns_are_jacobian_rows():
    """J^T e_k equals row k of J for nu~'s row and a momentum row, entry by
    entry against tangent columns over the nodes of k's two-ring."""
    print("[case] RANS-SA adjoint vs explicit Jacobian rows", flush=True)
    s, lv, u = make_rans(6, 2)
    n = u.shape[1]
    a, b = lv[0].side_index
    nbr = [set() for _ in range(n)]
    for p, q in zip(a, b):
        nbr[p].add(q)
        nbr[q].add(p)
    rng = np.random.default_rng(53)
    for node in rng.choice(n, 2, replace=False):
        ring = set(nbr[node]) | {node}
        ring2 = set().union(*(nbr[k] for k in ring)) | ring
        for comp in (5, 2):
            e = np.zeros((6, n))
            e[comp, node] = 1.0
            row = s.adjoint(e)
            for j in rng.choice(sorted(ring2), 4, replace=False):
                for c in range(6):
                    d = np.zeros((6, n))
                    d[c, j] = 1.0
                    t = s.tangent(d)[comp, node]
                    assert abs(t - row[c, j]) <= 1e-12 * (1 + abs(row[c, j])), (node, comp, j, c, t, row[c, j])
            # no entries outside the two-ring
            outside = np.ones(n, bool)
            outside[sorted(ring2)] = False
            assert np.all(row[:, outside] == 0.0)
    s.close()


@pytest.mark.parametrize("kind", ["euler2", "rans2"])
def test_device_vector_applies_equal_host_ones(kind):
    """flite_tangent_apply_device / flite_adjoint_apply_device on torch
    device tensors give the host entry points' results bit for bit, and
    host pointers are refused (before any device access)."""
    from flite3d_amd.device import DeviceError
    print(f"[case] device-vector applies {kind}", flush=True)
    if kind == "euler2":
        s, lv, u = make_smooth(8, 2)
        nc = 5
    else:
        s, lv, u = make_rans(8, 2)
        nc = 6
    n = lv[0].n_nodes
    x = np.random.default_rng(71).standard_normal((nc, n))
    for host, dev in ((s.tangent, s.tangent_device), (s.adjoint, s.adjoint_device)):
        ref = host(x)
        xd = torch.from_numpy(x.copy()).to("cuda:0")
        od = torch.zeros((nc, n), dtype=torch.float64, device="cuda:0")
        dev(xd.data_ptr(), od.data_ptr())
        assert np.array_equal(od.cpu().numpy(), ref)
    with pytest.raises(DeviceError):
        s.tangent_device(x.ctypes.data, x.ctypes.data)
    s.close()


@pytest.mark.parametrize("state", ["rest", "uniform"])
@pytest.mark.parametrize("order", [1, 2])
def test_rans_adjoint_dot_product_where_the_upwind_term_vanishes(order, state):
    """The SA convection's upwind term is exactly zero on a side whose ends
    are at rest, or whose weight is normal to a uniform flow, while nu~
    differs: tangent and adjoint take the same branch there too.  nu~'s row
    against the velocities and density holds the convection; the bar is that
    of the other states."""
    from cases import rans
    print(f"[case] RANS-SA adjoint at vanishing upwind terms order={order} {state}", flush=True)
    lv = levels(8, 2, jitter=0.0)
    iv = rans(hllcfluxorder=order, reynoldsnumber=1.0e4)
    s = Solver(iv.to_struct(), list(lv))
    s.init_freestream()
    inf = np.array(iv.inflowfield[0])
    x, y, z = lv[0].coords
    u = np.zeros((6, lv[0].n_nodes))
    u[0], u[4] = inf[0], inf[4]
    if state == "uniform":
        u[1] = inf[0]
    u[5] = 3.0 * (1.0 + 0.3 * np.sin(1.7 * x + 0.9 * y - 1.3 * z + 0.2))
    s.set(1, "U", u)
    s.apply(1, "PRESSURE")
    rng = np.random.default_rng(59)
    for rows, cols in [(range(6), range(6)), ([5], [0]), ([5], [1, 2, 3]), ([5], [5])]:
        du, lam = rng.standard_normal((2, 6, u.shape[1]))
        du[[c for c in range(6) if c not in cols]] = 0.0
        lam[[c for c in range(6) if c not in rows]] = 0.0
        terms = lam * s.tangent(du)
        a, b = np.sum(terms), np.sum(s.adjoint(lam) * du)
        scale = np.sqrt(np.sum(terms ** 2))
        assert abs(a - b) <= 1e-12 * max(abs(a), abs(b), scale), (list(rows), list(cols), a, b)
    s.close()
