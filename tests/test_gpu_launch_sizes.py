"""The passes a step is made of are chosen by the launch's size (row-split,
pipelined and plain kernels, with LDS halos); the batch option lds=0 keeps the
plain global-gather kernels at every size. All add in the same order, so state
and scalars must be the same bits on both sides of every size rule: one cell
block, partly filled slices and blocks, and the blocks around each limit."""
import numpy as np
import pytest

from nextgen_amd.batch import Batch, Instance, Layout
from nextgen_amd.ic import tgv_params
from nextgen_amd.ideal_gas import CG_PREC_FP64, CG_PREC_MIXED, Mesh, parse_params

from test_gpu_flux_passes import assert_same

pytestmark = pytest.mark.gpu

WALLS = ("y0 CBC_UPT 0.1 0.4 0 71.42857142857143 1.0\ny1 NSCBC_OUTLET_P 71.07 0.3 6.28\n")


def states(mesh, prec, text, lds):
    b = Batch(prec)
    b.set_option("lds", lds)
    b.set_option("graph", 0)
    x = Instance(mesh, parse_params(text), *mesh.ic_tgv(0.1, 1.4), layout=Layout(mesh, prec))
    i = b.attach(x)
    b.step(3)
    out = b.state(i), b.diag(i)
    b.close()
    return out


# cells (blocks of 256): 576 (3), 4080 (16), 16250 (64), 16900 (67), 47952 (188),
# 49284 (193), 97336 (381), 99452 (389), 262144 (1024), 266240 (1040)
@pytest.mark.parametrize("prec", [CG_PREC_FP64, CG_PREC_MIXED])
@pytest.mark.parametrize("kind,dims,sgs", [
    ("jittered", (9, 8, 8), "VREMAN"), ("jittered", (17, 16, 15), "SIGMA"), ("jittered", (26, 25, 25), "VREMAN"),
    ("jittered", (26, 26, 25), "NONE"), ("jittered", (37, 36, 36), "DSM_LOCAL"), ("jittered", (37, 37, 36), "VREMAN"),
    ("jittered", (46, 46, 46), "VREMAN"), ("jittered", (47, 46, 46), "VREMAN"), ("lattice", (64, 64, 64), "NONE"),
    ("lattice", (65, 64, 64), "NONE"), ("channel", (9, 11, 8), "VREMAN"), ("channel", (30, 28, 21), "VREMAN"),
    ("channel", (40, 38, 35), "NONE")])
def test_size_rules_bitwise(prec, kind, dims, sgs):
    if kind == "lattice":
        mesh = Mesh.lattice(dims)
    elif kind == "channel":
        mesh = Mesh.channel(dims, jitter=0.3, seed=5)
    else:
        mesh = Mesh.jittered(dims, 0.3, seed=5)
    text = tgv_params(sgs=sgs) + f"PRECISION {'MIXED' if prec == CG_PREC_MIXED else 'FP64'}\n"
    if kind == "channel":
        text += WALLS
    (a, da), (b, db) = states(mesh, prec, text, 1), states(mesh, prec, text, 0)
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)
    assert da.cfl_max == db.cfl_max and da.dt == db.dt


# blocks of 256 cells: 128, 132, 250; 250, 311, 326
@pytest.mark.parametrize("prec,dims,slices", [
    (CG_PREC_FP64, (32, 32, 32), True), (CG_PREC_FP64, (33, 32, 32), False), (CG_PREC_FP64, (40, 40, 40), False),
    (CG_PREC_MIXED, (40, 40, 40), True), (CG_PREC_MIXED, (43, 43, 43), True), (CG_PREC_MIXED, (44, 43, 44), False)])
def test_slice_halos_only_where_read(prec, dims, slices, monkeypatch):
    # the halos' share of a layout: 2 bytes per extended half-face (a twelfth more for
    # padding) and 4 bytes per halo cell (about four per cell) for the blocks; as much
    # again and about 25 bytes a cell for the slices of the row-split passes
    mesh = Mesh.jittered(dims, 0.3, seed=5)
    halves = 2 * (mesh.nef - mesh.nfa)
    with_halos = Layout(mesh, prec)
    monkeypatch.setenv("CG_NO_LDS", "1")
    without = Layout(mesh, prec)
    per_half = (with_halos.bytes() - without.bytes()) / halves
    assert 2.0 < per_half < 3.0 if not slices else 4.0 < per_half < 6.0


# the blocks around the row-split passes' limits: 128 and 132, 311 and 326
@pytest.mark.parametrize("kind", ["jittered", "lattice", "channel"])
@pytest.mark.parametrize("prec,dims", [("FP64", (32, 32, 32)), ("FP64", (33, 32, 32)), ("MIXED", (43, 43, 43)),
                                       ("MIXED", (44, 43, 44))])
def test_row_split_limit_bitwise(prec, dims, kind, monkeypatch):
    mesh = Mesh.lattice(dims) if kind == "lattice" else getattr(Mesh, kind)(dims, 0.3, 5)
    text = tgv_params(sgs="VREMAN") + f"PRECISION {prec}\n" + (WALLS if kind == "channel" else "")
    assert_same(monkeypatch, mesh, text, [{}])


# the scalar pass is compiled for 1, 2, 4 and 8 scalars: the counts that fill each and
# those that leave some unused, and a source (RES_TIME, by name the last here)
@pytest.mark.parametrize("prec", ["FP64", "MIXED"])
@pytest.mark.parametrize("kind,dims,count,res_time", [
    ("jittered", (9, 8, 8), 1, False), ("jittered", (9, 8, 8), 2, False), ("jittered", (17, 16, 15), 2, True),
    ("jittered", (13, 11, 10), 4, False), ("jittered", (13, 11, 10), 4, True), ("jittered", (17, 16, 15), 8, False),
    ("jittered", (12, 11, 9), 7, True), ("channel", (13, 11, 10), 2, False), ("channel", (13, 11, 10), 6, False),
    ("lattice", (11, 10, 9), 3, False), ("jittered", (30, 28, 21), 3, False),
    ("jittered", (40, 38, 36), 2, False), ("jittered", (66, 64, 63), 5, False)])
def test_scalar_counts_bitwise(kind, dims, count, res_time, prec, monkeypatch):
    if kind == "lattice":
        mesh = Mesh.lattice(dims)
    elif kind == "channel":
        mesh = Mesh.channel(dims, jitter=0.3, seed=9)
    else:
        mesh = Mesh.jittered(dims, 0.3, seed=9)
    text = tgv_params(sgs="VREMAN") + f"PRECISION {prec}\n" + "".join(f"REGISTER_SCALAR A{i}\n" for i in range(count))
    text += "RES_TIME\n" if res_time else ""
    if kind == "channel":
        inflow = "".join(f" A{i} {0.1 * (i + 1)}" for i in range(count))
        text += f"y0 CBC_UPT 0.1 0.4 0 71.42857142857143 1.0{inflow}\ny1 NSCBC_OUTLET_P 71.07 0.3 6.28\n"
    assert_same(monkeypatch, mesh, text, [{}, {"CG_TILE": "2"}])
