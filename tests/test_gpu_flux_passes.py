"""Which kernels a launch takes: the batch option "tile" (CG_TILE for a solver) at 2
and 8 runs the plain thread-per-cell LDS passes at every size, at its default the
passes are chosen by the launch's size. Every choice gives the bits of the global
gathers (lds=0, CG_NO_LDS): with each boundary type, in each
layout order, for a step and for a right-hand side alone.

The kernels are read from a trace of the launches, taken in a process of its own so
that the tracer stays out of the other tests.
"""
import json
import os
import subprocess
import sys

import numpy as np
import pytest

from nextgen_amd.batch import Batch
from nextgen_amd.ic import tgv_params
from nextgen_amd.ideal_gas import CG_PREC_FP64, CG_PREC_MIXED, IdealGasSolver, Mesh, parse_params

from test_gpu_walls import WALLS as BOUNDARIES, channel_state, deck

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

TRACE = """
import json, os, re, sys
import torch
from torch.profiler import ProfilerActivity, profile
from nextgen_amd.batch import Batch
from nextgen_amd.ic import tgv_params
from nextgen_amd.ideal_gas import IdealGasSolver, Mesh, parse_params

torch.zeros(1, device="cuda")


def kernels(fn):
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        fn()
        torch.cuda.synchronize()
    return [e.key.replace("void (anonymous namespace)::", "").split("(")[0] for e in p.key_averages()
            if "::k_" in e.key]


out = []
for dims, prec, tile in json.loads(sys.argv[1]):
    m = Mesh.lattice(dims)
    p = parse_params(tgv_params(sgs="NONE") + "PRECISION " + ("MIXED" if prec else "FP64") + "\\n")
    b = Batch(prec)
    b.set_option("graph", 0)
    b.set_option("tile", tile)
    b.add(m, p, *m.ic_tgv(0.1, 1.4))
    batch = kernels(lambda: b.step(1))
    b.close()
    os.environ["CG_TILE"] = str(tile)
    s = IdealGasSolver(m, p)
    s.set_state(*m.ic_tgv(0.1, 1.4))
    s.init_complete()
    solver = kernels(lambda: s.advance_solution(1))
    s.close()
    out.append([batch, solver])
# tuned while large, then shrunk
for prec in (0, 1):
    p = parse_params(tgv_params(sgs="NONE") + "PRECISION " + ("MIXED" if prec else "FP64") + "\\n")
    b = Batch(prec)
    b.set_option("graph", 0)
    ids = [b.add(m, p, *m.ic_tgv(0.1, 1.4)) for m in (Mesh.lattice((65, 64, 64)), Mesh.lattice(12))]
    b.tune(2)
    b.remove(ids[0])
    b.step(1)
    out.append([kernels(lambda: b.step(1)), b.tune(2).splitlines()[-1], b.tune(2).splitlines()[-1]])
    b.close()
print("TRACE " + json.dumps(out))
"""

# (dims, precision, tile, flux pass, its last template value or None, properties pass)
R, P, L = "k_flux_rows", "k_flux_pipe", "k_flux_lds"
ROUTES = [
    ((12, 12, 12), CG_PREC_FP64, 2, L, 2, "k_props"), ((12, 12, 12), CG_PREC_FP64, 8, L, 8, "k_props"),
    ((12, 12, 12), CG_PREC_MIXED, 2, L, 2, "k_props"), ((12, 12, 12), CG_PREC_MIXED, 8, L, 8, "k_props"),
    ((40, 40, 40), CG_PREC_FP64, 8, L, 8, "k_props"), ((48, 48, 48), CG_PREC_MIXED, 2, L, 2, "k_props"),
    # the limits of the row-split passes (128 blocks of 256 cells in FP64, 320 in mixed
    # precision; ten wavefronts up to 64) and of the pipelined one (1024)
    ((32, 32, 16), CG_PREC_FP64, 4, R, 10, "k_props_rows"), ((33, 32, 16), CG_PREC_FP64, 4, R, 5, "k_props_rows"),
    ((32, 32, 32), CG_PREC_FP64, 4, R, 5, "k_props_rows"), ((33, 32, 32), CG_PREC_FP64, 4, P, None, "k_props"),
    ((64, 40, 32), CG_PREC_MIXED, 4, R, 5, "k_props_rows"), ((65, 40, 32), CG_PREC_MIXED, 4, P, None, "k_props"),
    ((64, 64, 64), CG_PREC_FP64, 4, P, None, "k_props"), ((65, 64, 64), CG_PREC_FP64, 4, L, 4, "k_props"),
    ((64, 64, 64), CG_PREC_MIXED, 4, P, None, "k_props"), ((65, 64, 64), CG_PREC_MIXED, 4, L, 4, "k_props"),
]


@pytest.fixture(scope="module")
def traces():
    r = subprocess.run([sys.executable, "-c", TRACE, json.dumps([t[:3] for t in ROUTES])], cwd=ROOT,
                       capture_output=True, text=True, timeout=110)
    assert r.returncode == 0, r.stderr[-2000:]
    line = [x for x in r.stdout.splitlines() if x.startswith("TRACE ")][-1]
    return json.loads(line[6:])


# a batch tuned beyond the pipelined pass, whichever tile was kept there, takes the
# passes of its size once solves have left; those do not read the tile, and the tuner
# leaves it alone
@pytest.mark.parametrize("prec", [0, 1])
def test_tuned_batch_that_shrinks(traces, prec):
    names, again, once_more = traces[len(ROUTES) + prec]
    assert [n.split("<")[0] for n in names if n.startswith("k_flux")] == [R] * 3, names
    assert again.split("tile")[1] == once_more.split("tile")[1]


def route_id(i):
    dims, prec, tile = ROUTES[i][:3]
    return "x".join(map(str, dims)) + ("-mixed" if prec == CG_PREC_MIXED else "-fp64") + f"-tile{tile}"


@pytest.mark.parametrize("i", range(len(ROUTES)), ids=route_id)
def test_kernels_of_a_step(traces, i):
    _, _, _, flux, last, props = ROUTES[i]
    for names in traces[i]:
        ran = [n for n in names if n.startswith("k_flux")]
        assert len(ran) == 3 and all(n.split("<")[0] == flux for n in ran), names
        if last is not None:
            assert all(n.rstrip(">").split(",")[-1].strip() == str(last) for n in ran), ran
        assert [n.split("<")[0] for n in names if n.startswith("k_props")] == [props], names


WALLS = "y0 CBC_UPT 0.1 0.4 0 71.42857142857143 1.0\ny1 NSCBC_OUTLET_P 71.07 0.3 6.28\n"


@pytest.mark.parametrize("prec", [CG_PREC_FP64, CG_PREC_MIXED])
@pytest.mark.parametrize("kind,sgs", [("jittered", "DSM_LOCAL"), ("channel", "VREMAN")])
def test_tile_bitwise(prec, kind, sgs):
    dims = (13, 11, 10)
    mesh = Mesh.channel(dims, jitter=0.3, seed=7) if kind == "channel" else Mesh.jittered(dims, 0.3, seed=7)
    text = tgv_params(sgs=sgs) + f"PRECISION {'MIXED' if prec == CG_PREC_MIXED else 'FP64'}\n"
    text += WALLS if kind == "channel" else ""
    runs = []
    for option, value in (("lds", 0), ("tile", 2), ("tile", 8), ("tile", 4)):
        b = Batch(prec)
        b.set_option(option, value)
        i = b.add(mesh, parse_params(text), *mesh.ic_tgv(0.1, 1.4))
        b.step(4)
        runs.append(b.state(i))
        b.close()
    for run in runs[1:]:
        for x, y in zip(run, runs[0]):
            np.testing.assert_array_equal(x, y)


def solve(monkeypatch, mesh, text, env, nsteps=3):
    """State, right-hand side, scalars, dt and CFL maximum after nsteps, under env."""
    for k in ("CG_NO_LDS", "CG_TILE", "CG_LANE_ORDER", "CG_CELL_ORDER"):
        monkeypatch.delenv(k, raising=False)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    x = mesh.get("x_cv")
    s = IdealGasSolver(mesh, parse_params(text))
    s.set_state(*(channel_state(mesh) if mesh.nbf else mesh.ic_tgv(0.1, 1.4)))
    for i, name in enumerate(n for n in s.scalar_names() if n != "RES_TIME"):
        s.set_scalar(name, 0.5 + 0.5 * np.sin((i + 1) * x[:, 0] + x[:, 2]) * np.cos(x[:, 1]))
    s.init_complete()
    s.advance_solution(nsteps)
    d = s.report()
    out = [*s.get_state(), s.calc_rhs(1), *(s.get_scalar(n) for n in s.scalar_names()), np.array([d.dt, d.cfl_max])]
    s.close()
    assert all(np.isfinite(v).all() for v in out)
    return out


def assert_same(monkeypatch, mesh, text, envs):
    ref = solve(monkeypatch, mesh, text, {"CG_NO_LDS": "1"})
    for env in envs:
        got = solve(monkeypatch, mesh, text, env)
        assert len(got) == len(ref)
        for a, b in zip(got, ref):
            np.testing.assert_array_equal(a, b, err_msg=str(env))


# the row-split passes and the plain one
@pytest.mark.parametrize("prec", ["FP64", "MIXED"])
@pytest.mark.parametrize("walls", sorted(BOUNDARIES))
def test_boundary_types_bitwise(walls, prec, monkeypatch):
    mesh = Mesh.channel((13, 11, 10), jitter=0.3, seed=7)
    assert_same(monkeypatch, mesh, deck(BOUNDARIES[walls], prec=prec), [{}, {"CG_TILE": "2"}, {"CG_TILE": "8"}])


# the pipelined pass: 208 blocks in FP64, 389 in mixed precision
@pytest.mark.parametrize("prec,dims", [("FP64", (40, 38, 35)), ("MIXED", (48, 46, 45))])
@pytest.mark.parametrize("walls", ["cbc_upt+sponge", "nscbc_mt_t0+nscbc", "wmeqiso+wmeqiso"])
def test_boundary_types_pipelined_bitwise(walls, prec, dims, monkeypatch):
    mesh = Mesh.channel(dims, jitter=0.3, seed=7)
    assert_same(monkeypatch, mesh, deck(BOUNDARIES[walls], prec=prec), [{}])


# beyond the pipelined pass: 1040 blocks
@pytest.mark.parametrize("prec", ["FP64", "MIXED"])
def test_large_channel_bitwise(prec, monkeypatch):
    mesh = Mesh.channel((65, 64, 64), jitter=0.3, seed=7)
    assert_same(monkeypatch, mesh, deck(BOUNDARIES["cbc_upt+nscbc"], prec=prec), [{}, {"CG_TILE": "8"}])


# layouts in which a slice's first lane need not have the most half-faces: rows past a
# lane's last read a slot that may be padding
@pytest.mark.parametrize("prec", ["FP64", "MIXED"])
@pytest.mark.parametrize("dims,sgs,count", [((12, 11, 10), "DSM_LOCAL", 3), ((47, 46, 46), "DSM_LOCAL", 1),
                                            ((66, 64, 63), "SIGMA", 0)])
def test_layout_orders_every_pass_bitwise(dims, sgs, count, prec, monkeypatch):
    mesh = Mesh.jittered(dims, 0.3, seed=11)
    text = tgv_params(sgs=sgs) + f"PRECISION {prec}\n" + "".join(f"REGISTER_SCALAR Z{i}\n" for i in range(count))
    orders = [{"CG_LANE_ORDER": "plain"}, {"CG_CELL_ORDER": "sorted256", "CG_LANE_ORDER": "plain"},
              {"CG_CELL_ORDER": "sorted64"}]
    orders = orders if dims[0] < 40 else orders[:2]
    assert_same(monkeypatch, mesh, text, orders + [{**o, "CG_TILE": "2"} for o in orders if dims[0] < 40])
