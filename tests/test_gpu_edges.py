"""Sizes at which a launch shape or a kernel's split changes, on the GPU
against the oracle, and the lanes-per-node variants of the linearised
kernels against each other.

Bars as in test_gpu_parity: 1e-11 of the component scale for single
operations, 1e-9 for states after whole V-cycles, 1e-8 for monitor sums and
forces.  The lanes of the linearised kernels only change the order of sums of
at most a few dozen terms, each combined once per stage of the chain, so their
results are held to the single operations' 1e-11.
"""
import ctypes
import dataclasses
import math

import numpy as np
import pytest

from flite3d_amd.device import Solver, lib

from cases import euler, levels, rans
from test_gpu_parity import jst_case, pair, perturb, rel_err

pytestmark = pytest.mark.gpu


def cycles_match(iv, lv, n=3):
    s, o = pair(iv, lv)
    s.init_freestream(); o.init_freestream()
    for c in range(1, n + 1):
        s.cycle(c); o.cycle(c)
    ms, mo = s.monitor(), o.monitor()
    assert np.allclose(ms["res"], mo["res"], rtol=1e-8, atol=1e-16), (ms["res"], mo["res"])
    assert np.allclose(ms["forces"], mo["forces"], rtol=1e-8, atol=1e-14), (ms["forces"], mo["forces"])
    nc = 6 if iv.turbulencemodel == 1 else 5
    e = rel_err(s.get(1, "U")[:nc], o.get(1, "U")[:nc])
    s.close(); o.close()
    assert e.max() < 1e-9, e


@pytest.mark.parametrize("n,nl", [(2, 1), (3, 2), (4, 2), (9, 3), (17, 3)])
@pytest.mark.parametrize("kind", ["euler1", "euler2", "rans"])
def test_cycles_at_block_remainders(kind, n, nl):
    """The smallest meshes (less than one wavefront of nodes), node and side
    blocks with remainders on each level, and 324 wall nodes (n = 17), beyond
    the force integral's one-wavefront order."""
    print(f"[case] {kind} n={n} levels={nl}", flush=True)
    iv = rans(multigridscheme=3) if kind == "rans" else euler(int(kind[-1]), multigridscheme=3)
    cycles_match(iv, levels(n, nl, first_cell=0.01 if kind == "rans" else None))


@pytest.mark.parametrize("n", [25, 40])
def test_first_order_stage_rule(n):
    """Both sides of the size rule of the one-launch first-order stage without
    a turbulence equation (17.6k and 68.9k level-1 nodes): the state after two
    cycles as the oracle has it."""
    print(f"[case] first-order stage rule n={n}", flush=True)
    cycles_match(euler(1, multigridscheme=3), levels(n, 2), 2)


@pytest.mark.parametrize("lanes", ["1", "4", "16"])
@pytest.mark.parametrize("name", ["llf", "roe_matrix"])
def test_jst_lanes(name, lanes, monkeypatch):
    print(f"[case] jst {name} lanes {lanes}", flush=True)
    monkeypatch.setenv("FLITE_GATHER_LANES", lanes)
    s, o = pair(jst_case(name), levels(9, 2))
    s.init_freestream(); o.init_freestream()
    perturb(s, o, 1, np.random.default_rng(5), amp=0.05)
    for x in (s, o):
        x.apply(1, "PRESSURE_ABS")
        x.apply(1, "TIMESTEPS")
        x.apply(1, "DISSIPATION")
        x.apply(1, "RHS")
    for f in ("DT", "DISSIPATION", "RHS"):
        e = rel_err(s.get(1, f), o.get(1, f))
        assert e.max() < 1e-11, (f, e)
    s.close(); o.close()


@pytest.mark.parametrize("order,fp32", [(1, False), (2, True)])
def test_fields_round_trip(order, fp32):
    """Fields renumbered on the device come back as they went in, on each
    level: bit for bit in FP64, as the nearest FP32 on FP32 levels."""
    print(f"[case] field round trip order={order} fp32={fp32}", flush=True)
    lv = levels(9, 3)
    s, o = pair(euler(order), lv, fp32)
    o.close()
    s.init_freestream()
    rng = np.random.default_rng(8)
    for k in range(1, 4):
        u = s.get(k, "U")
        u = u * (1.0 + 0.1 * rng.uniform(-1, 1, size=u.shape))
        s.set(k, "U", u)
        want = u.astype(np.float32).astype(np.float64) if fp32 and k > 1 else u
        assert np.array_equal(s.get(k, "U")[:5], want[:5]), k
    s.close()


@pytest.mark.parametrize("kind", ["euler1", "euler2", "rans1", "rans2"])
def test_linearised_lanes(kind, monkeypatch):
    print(f"[case] linearised lanes {kind}", flush=True)
    order = int(kind[-1])
    sa = kind.startswith("rans")
    iv = rans(hllcfluxorder=order) if sa else euler(order)
    lv = levels(9, 1, first_cell=0.01 if sa else None)
    nc = 6 if sa else 5
    got = {}
    for lanes in ("1", "4", "16"):
        monkeypatch.setenv("FLITE_GATHER_LANES", lanes)
        s = Solver(iv.to_struct(), list(lv))
        s.init_freestream()
        rng = np.random.default_rng(9)
        u = s.get(1, "U")
        u = u * (1.0 + 0.02 * rng.uniform(-1, 1, size=u.shape))
        if sa:
            u[5] = 0.1 + 5.0 * rng.uniform(0, 1, size=u.shape[1])
        s.set(1, "U", u)
        s.apply(1, "PRESSURE")
        v = rng.standard_normal((nc, u.shape[1]))
        got[lanes] = s.tangent(v), s.adjoint(v)
        s.close()
    for lanes in ("1", "4"):
        for a, b in zip(got[lanes], got["16"]):
            assert np.abs(b).max() > 0
            e = rel_err(a, b)
            assert e.max() < 1e-11, (lanes, e)


@pytest.mark.parametrize("order", [1, 2])
def test_cycle_without_smoothing_steps(order):
    """numberOfRelaxationSteps 0: the transfers alone, from a state and time
    steps that one smoothing step left.  The restricted state keeps the
    pressure the restriction formed, which the prolongation's far field reads."""
    print(f"[case] no smoothing steps, order={order}", flush=True)
    iv = euler(order, multigridscheme=1, numberofrelaxationsteps=0)
    s, o = pair(iv, levels(8, 3))
    s.init_freestream(); o.init_freestream()
    perturb(s, o, 1, np.random.default_rng(3), amp=0.05)
    for x in (s, o):
        x.do_time_iterations(1, 1, True)
        x.cycle(1)
        x.cycle(2)
    for k in (1, 2, 3):
        for f in ("U", "PRESSURE"):
            e = rel_err(s.get(k, f)[:5], o.get(k, f)[:5])
            assert e.max() < 1e-9, (k, f, e)
    s.close(); o.close()


@pytest.mark.parametrize("name", ["llf", "roe"])
@pytest.mark.parametrize("level", [1, 2])
def test_jst_reads_the_stored_momenta(name, level):
    """Equal momenta on unequal densities: the dissipation's momentum
    differences are exactly zero."""
    print(f"[case] jst momenta {name} level={level}", flush=True)
    s, o = pair(jst_case(name), levels(8, 2))
    o.close()
    s.init_freestream()
    rng = np.random.default_rng(12)
    u = s.get(level, "U")
    u[0] = rng.uniform(0.8, 1.2, u.shape[1])
    u[1:4] = np.array([0.7, 0.3, -0.2])[:, None]
    s.set(level, "U", u)
    for op in ("PRESSURE", "TIMESTEPS", "DISSIPATION"):
        s.apply(level, op)
    d = s.get(level, "DISSIPATION")
    s.close()
    assert np.abs(d[0]).max() > 0
    assert np.all(d[1:4] == 0.0), np.abs(d[1:4]).max()


def test_central_flux_reads_the_stored_momenta():
    """Side weights and momenta of few bits, unequal densities: the central
    mass fluxes and their sums are exact, away from the boundary sides."""
    print("[case] central flux momenta", flush=True)
    lv = levels(8, 1)
    w = np.round(lv[0].side_w * 2.0 ** 20) / 2.0 ** 20
    lv = [dataclasses.replace(lv[0], side_w=w)]
    s = Solver(jst_case("central").to_struct(), lv)
    s.init_freestream()
    rng = np.random.default_rng(13)
    u = s.get(1, "U")
    m = np.array([0.75, 0.25, -0.375])
    u[0] = rng.uniform(0.8, 1.2, u.shape[1])
    u[1:4] = m[:, None]
    s.set(1, "U", u)
    s.apply(1, "PRESSURE")
    s.apply(1, "RHS")
    r = s.get(1, "RHS")[0]
    s.close()
    want = np.zeros(u.shape[1])
    f = 2.0 * (m @ w)
    base = lv[0].side_index.min()
    a, b = lv[0].side_index - base
    np.add.at(want, a, f)
    np.add.at(want, b, -f)
    inner = np.ones(u.shape[1], bool)
    inner[lv[0].bside_index[:2] - base] = False
    assert inner.sum() > 100 and np.abs(want[inner]).max() > 0
    assert np.array_equal(r[inner], want[inner]), np.abs(r - want)[inner].max()


def free_device_memory():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_field_access_takes_no_device_memory():
    """Fields of any width go through the context's own staging: reading 25
    components of 68.9k nodes (14 MB) leaves the device's free memory as it
    was."""
    print("[case] field access and device memory", flush=True)
    s = Solver(euler(2).to_struct(), list(levels(40, 1)))
    s.init_freestream()
    s.cycle(1)
    s.get(1, "PRESSURE")
    before = free_device_memory()
    g = s.get(1, "GRADIENT")
    s.set(1, "U", s.get(1, "U"))
    after = free_device_memory()
    s.close()
    assert g.shape[0] == 25 and np.abs(g[:15]).max() > 0
    assert after == before, before - after


@pytest.mark.parametrize("kind", ["euler1", "jst", "rans"])
def test_autotune_times_the_cycle(kind, monkeypatch):
    """Autotuning times the launches a cycle makes.  Where no launch of a
    level depends on its lanes (the one-launch stages with their time steps)
    the lanes stay as they were; elsewhere one lane a node, the slowest on
    levels this small, gives way.  The cycles that follow are the oracle's."""
    print(f"[case] autotune {kind}", flush=True)
    monkeypatch.setenv("FLITE_GATHER_LANES", "1")
    iv = {"euler1": euler(1, multigridscheme=3), "jst": jst_case("roe", multigridscheme=3),
          "rans": rans(multigridscheme=3)}[kind]
    s, o = pair(iv, levels(8, 2, first_cell=0.005 if kind == "rans" else None))
    s.init_freestream(); o.init_freestream()
    lanes = s.autotune(5)
    assert lanes == [1, 1] if kind == "euler1" else lanes[0] in (4, 16), lanes
    for c in (1, 2):
        s.cycle(c); o.cycle(c)
    e = rel_err(s.get(1, "U")[:5], o.get(1, "U")[:5])
    s.close(); o.close()
    assert e.max() < 1e-9, e


@pytest.mark.parametrize("lanes", ["1", "4", "16"])
def test_gradient_rounds_the_differences(lanes, monkeypatch):
    """The Green-Gauss sums' rounding is one of the neighbours' differences,
    not of the values, whatever the lanes: against extended precision, at most
    (terms + 4) 2^-53 of the sum of |differences times weights| with up to 40
    terms a node, hence 32 x 2^-52 of it."""
    print(f"[case] gradient rounding lanes={lanes}", flush=True)
    monkeypatch.setenv("FLITE_GATHER_LANES", lanes)
    lv = levels(9, 1)
    s = Solver(euler(2).to_struct(), list(lv))
    s.init_freestream()
    x, y, z = lv[0].coords
    u = s.get(1, "U")
    wave = np.sin(1.3 * x + 0.7 * y - 0.9 * z)
    u[0] = 1.0 + 1e-3 * wave
    u[1:4] = u[0] * np.array([0.9, 0.1, 0.2])[:, None] * (1.0 + 1e-3 * wave)
    u[4] = 1e3 + 1e-2 * wave
    s.set(1, "U", u)
    s.apply(1, "PRESSURE")
    s.apply(1, "RHS")
    got = s.get(1, "GRADIENT")[:15].reshape(3, 5, -1)
    s.close()
    q = np.concatenate([u[:1], u[1:4] / u[0], u[4:5]]).astype(np.longdouble)
    base = lv[0].side_index.min()
    a, b = lv[0].side_index - base
    ba, bb = lv[0].bside_index[:2] - base
    want, size = np.zeros((2, 3, 5, u.shape[1]), np.longdouble)
    for d in range(3):
        w, wb = lv[0].side_w[d].astype(np.longdouble), lv[0].bside_w[d].astype(np.longdouble)
        terms = [[] for _ in range(u.shape[1])]  # a node's weights cancel: summed exactly
        for node, sign, weight in ((a, 1, w), (b, -1, w), (ba, 2, wb), (bb, 2, wb)):
            for k, v in zip(node, sign * weight):
                terms[k].append(float(v))
        own = np.array([math.fsum(t) for t in terms], np.longdouble)
        for c in range(5):
            for i, j, weight in ((a, b, w), (b, a, -w), (ba, bb, wb), (bb, ba, wb)):
                np.add.at(want[d, c], i, (q[c][j] - q[c][i]) * weight)
                np.add.at(size[d, c], i, abs((q[c][j] - q[c][i]) * weight))
            want[d, c] += 2 * q[c] * own
            size[d, c] += abs(2 * q[c] * own)
    vol = lv[0].volume.astype(np.longdouble)
    e = abs(got - want / vol) / (size / vol)
    assert np.abs(want).max() > 0
    assert e.max() <= 32 * 2.0 ** -52, e.max()


@pytest.mark.parametrize("env", [{"FLITE_FLUX_KERNEL": "block"},
                                 {"FLITE_FLUX_KERNEL": "block", "FLITE_SIDE_BLOCK": "512"}])
@pytest.mark.parametrize("kind", ["euler1", "rans"])
def test_first_order_side_blocks(kind, env, monkeypatch):
    """Side blocks of both shapes on the first-order levels, which run their
    stages in one launch unless told otherwise."""
    print(f"[case] first-order side blocks {kind} {env}", flush=True)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    iv = rans(multigridscheme=3) if kind == "rans" else euler(1, multigridscheme=3)
    cycles_match(iv, levels(8, 3, first_cell=0.005 if kind == "rans" else None))


@pytest.mark.parametrize("n", [24, 25])
def test_first_order_stage_rule_with_sa(n):
    """Both sides of the one-launch stage's size rule with a turbulence
    equation (15.6k and 17.6k level-1 nodes)."""
    print(f"[case] first-order SA stage rule n={n}", flush=True)
    cycles_match(rans(hllcfluxorder=1, multigridscheme=3), levels(n, 2, first_cell=0.005), 2)
