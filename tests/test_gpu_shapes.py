"""The kernels at the shapes where their splits of the work can go wrong, against the oracle
on the same tree: f64 within 1e-12 (the sums' order and 2^-53 per term, amplified by at most
the M2L's cancellation), the mixed precision within 1e-6."""
import sys

import numpy as np
import pytest

import fmm_amd
from fmm_amd import tune
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _log(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if fmm_amd.device_count() < 1:
        pytest.skip("no GPU")


def _check(fmm, ref, q, gradients=True, tol=1e-12):
    out = fmm.evaluate(q)
    phi, grad = ref.evaluate(q)
    errs = [O.error_norms(out.potential, phi)[0]]
    if gradients:
        errs.append(O.error_norms(out.gradient, grad, True)[0])
    _log(f"  errors {errs}")
    assert max(errs) < tol, errs
    again = fmm.evaluate(q)
    assert np.array_equal(out.potential, again.potential)


@pytest.mark.parametrize("p,leaf,gradients", [(0, 3, True), (1, 5, False), (4, 70, True), (9, 150, False),
                                              (14, 64, True), (15, 33, True), (15, 9, False)])
def test_m2p_rows_over_waves(p, leaf, gradients):
    """Long W rows (a dense cluster beside large leaves), leaves of one target to several
    passes of targets, the degrees where a workgroup holds fewer than eight waves."""
    _log(f"case M2P rows p={p} leaf={leaf} gradients={gradients}")
    rng = O.Rng(77)
    pts = np.vstack([rng.plummer(1500, (0.5, 0.5, 0.5), 0.01), rng.cube(600)])
    q = rng.normals(len(pts))
    fmm = fmm_amd.FmmBuilder(p).max_points_per_leaf(leaf).gradients(gradients).build(pts)
    rows = [len(fmm.plan.list("w", level)[1]) for level in range(fmm.plan.nlevels)]
    assert sum(rows) > 0
    _check(fmm, O.Fmm(pts, p=p, leaf_points=leaf, gradients=gradients), q, gradients)


def _class_rows(plan, p, precision):
    """The boxes whose M2L runs by reflection classes."""
    return sum(int(np.count_nonzero(np.diff(plan.list("v", level)[0])))
               for level in tune.m2l_class_levels(plan, p, precision))


@pytest.mark.parametrize("precision,tol", [("f64", 1e-12), ("mixed", 1e-6)])
@pytest.mark.parametrize("p", [0, 1, 4, 5, 6, 8, 10, 11, 12, 13, 14, 15])
def test_m2l_reflection_classes(p, precision, tol):
    """Dense levels at every count of row tiles (1 to 20) and of coefficient chunks, boundary
    boxes (sources missing at some reflections), target rows that do not fill a workgroup."""
    _log(f"case M2L reflection p={p} {precision}")
    rng = O.Rng(91 + p)
    pts = np.vstack([rng.cube(4500), rng.plummer(1500, (0.4, 0.6, 0.5), 0.03)])
    q = rng.normals(len(pts))
    fmm = fmm_amd.FmmBuilder(p).max_points_per_leaf(24).precision(precision).build(pts)
    rows = _class_rows(fmm.plan, p, precision)
    assert 0 < rows < 512 * 16  # less than a round of workgroups: every row through scratch rows
    _check(fmm, O.Fmm(pts, p=p, leaf_points=24), q, tol=tol)


@pytest.mark.parametrize("precision,tol", [("f64", 1e-12), ("mixed", 1e-6)])
@pytest.mark.parametrize("p", [4, 7, 12])
def test_m2l_reflection_whole_rounds(p, precision, tol):
    """More than a round of workgroups (1,024 of 16 boxes in f64, 512 of 32 mixed): the rows of the
    whole rounds add to the locals themselves, those of the last go through scratch rows.  Against
    the rotation M2L in f64, another path from the multipoles to the locals."""
    _log(f"case M2L reflection, whole rounds p={p} {precision}")
    rng = O.Rng(92)
    pts = rng.cube(60000)
    q = rng.normals(len(pts))
    plan = fmm_amd.Plan(pts, leaf_points=8)
    rows = _class_rows(plan, p, precision)
    assert rows > 16384 and rows % 16384 != 0
    out = fmm_amd.Fmm(plan, fmm_amd.Operator(plan, p, precision)).evaluate(q)
    ref = fmm_amd.Fmm(plan, fmm_amd.Operator(plan, p, "f64", m2l="rotation")).evaluate(q)
    errs = [O.error_norms(out.potential, ref.potential)[0], O.error_norms(out.gradient, ref.gradient, True)[0]]
    _log(f"  errors {errs}")
    assert max(errs) < tol, errs


@pytest.mark.parametrize("points,every", [(1000, False), (20000, True)])
def test_m2l_class_tables_of_an_operator(tmp_path, points, every):
    """The M2L tables that an operator builds (the classes' alone where no level takes a
    contraction, all with a level that does), built, stored and loaded: the same bits."""
    _log(f"case M2L class tables, {points} points")
    rng = O.Rng(93)
    pts = rng.cube(points)
    q = rng.normals(points)
    plan = fmm_amd.Plan(pts, leaf_points=8)
    classes = tune.m2l_class_levels(plan, 6, "f64")
    others = [l for l in range(2, plan.nlevels) if len(plan.list("v", l)[1]) and l not in classes]
    assert classes and bool(others) == every
    out = []
    try:
        for directory in (None, tmp_path, tmp_path):
            fmm_amd.set_table_cache(directory)
            out.append(fmm_amd.Fmm(plan, fmm_amd.Operator(plan, 6, "f64")).evaluate(q))
        assert fmm_amd.table_cache_stats() == (1, 0)
    finally:
        fmm_amd.set_table_cache(None)
    ref = fmm_amd.Fmm(plan, fmm_amd.Operator(plan, 6, "f64", m2l="rotation")).evaluate(q)
    assert O.error_norms(out[0].potential, ref.potential)[0] < 1e-12
    for o in out[1:]:
        assert np.array_equal(o.potential, out[0].potential) and np.array_equal(o.gradient, out[0].gradient)


@pytest.mark.parametrize("precision", ["f64", "mixed"])
def test_m2l_reflection_level_calls(precision):
    """The level calls run each level's share of the tasks (whole and split into parts)."""
    _log(f"case M2L reflection, level by level {precision}")
    rng = O.Rng(92)
    pts = rng.cube(60000)
    q = rng.normals(len(pts))
    fmm = fmm_amd.FmmBuilder(7).max_points_per_leaf(8).precision(precision).build(pts)
    assert _class_rows(fmm.plan, 7, precision) > 16384
    a, b = fmm.evaluate(q), fmm.evaluate_levels(q)
    assert O.error_norms(b.potential, a.potential)[0] < 1e-14
    assert O.error_norms(b.gradient, a.gradient, True)[0] < 1e-14


@pytest.mark.parametrize("precision,tol", [("f64", 1e-12), ("mixed", 2e-6)])
@pytest.mark.parametrize("k,leaf,gradients", [(9.0, 5, True), (2.0 + 0.5j, 40, True), (30.0, 70, False),
                                              (14.0, 150, True)])
def test_helmholtz_p2p_rows_over_waves(k, leaf, gradients, precision, tol):
    """Leaves of one target to several chunks of 128 (one or two targets per lane), rows of one
    near leaf to many, phases k r of many turns; real and complex wavenumbers."""
    _log(f"case Helmholtz P2P k={k} leaf={leaf} {precision} gradients={gradients}")
    rng = O.Rng(55)
    pts = np.vstack([rng.cube(900), rng.plummer(700, (0.5, 0.5, 0.5), 0.02)])
    q = rng.normals(len(pts)) + 1j * rng.normals(len(pts))
    b = fmm_amd.HelmholtzFmmBuilder(k, degree=10).max_points_per_leaf(leaf).gradients(gradients).precision(precision)
    fmm = b.build(pts)
    out = fmm.evaluate(q)
    phi, grad = O.Fmm(pts, p=10, leaf_points=leaf).evaluate_helmholtz(k, q)
    errs = [np.linalg.norm(out.potential - phi) / np.linalg.norm(phi)]
    if gradients:
        errs.append(np.linalg.norm(out.gradient - grad) / np.linalg.norm(grad))
    _log(f"  errors {errs}")
    assert max(errs) < tol, errs


@pytest.mark.parametrize("precision,tol", [("f64", 1e-12), ("mixed", 2e-6)])
@pytest.mark.parametrize("p,k", [(5, 3.0 + 0.2j), (9, 6.0)])
def test_helmholtz_m2l_reflection_classes(p, k, precision, tol):
    """Complex tables as two sets, a level at a time, over 100,000 pairs."""
    _log(f"case Helmholtz M2L reflection p={p} k={k} {precision}")
    rng = O.Rng(56)
    pts = np.vstack([rng.cube(9000), rng.plummer(1000, (0.5, 0.5, 0.5), 0.02)])
    q = rng.normals(len(pts)) + 1j * rng.normals(len(pts))
    b = fmm_amd.HelmholtzFmmBuilder(k, degree=p).max_points_per_leaf(10).precision(precision)
    fmm = b.build(pts)
    assert sum(len(fmm.plan.list("v", level)[1]) for level in range(2, fmm.plan.nlevels)) >= 100_000
    # (a table for each offset would be twice what the operator holds)
    per_offset = [len(np.unique(fmm.plan.list("v", level)[2])) for level in range(2, fmm.plan.nlevels)]
    _log(f"  {fmm.operator.stats()['device_bytes']} bytes, tables per offset {sum(per_offset) * 2 * (p + 1) ** 4 * 8}")
    out = fmm.evaluate(q)
    phi, grad = O.Fmm(pts, p=p, leaf_points=10).evaluate_helmholtz(k, q)
    errs = [np.linalg.norm(out.potential - phi) / np.linalg.norm(phi),
            np.linalg.norm(out.gradient - grad) / np.linalg.norm(grad)]
    _log(f"  errors {errs}")
    assert max(errs) < tol, errs


@pytest.mark.parametrize("precision,tol", [("f64", 1e-12), ("mixed", 2e-6)])
def test_helmholtz_small_trees_take_the_classes(precision, tol):
    """A tree of few pairs holds 56 offsets' tables a level, not one for each of its offsets."""
    p, k = 10, 25.0
    _log(f"case Helmholtz M2L reflection on a small tree {precision}")
    rng = O.Rng(58)
    pts = rng.cube(3000)
    q = rng.normals(len(pts)) + 1j * rng.normals(len(pts))
    fmm = fmm_amd.HelmholtzFmmBuilder(k, degree=p).max_points_per_leaf(40).precision(precision).build(pts)
    per_offset = [len(np.unique(fmm.plan.list("v", level)[2])) for level in range(2, fmm.plan.nlevels)]
    assert 0 < sum(len(fmm.plan.list("v", level)[1]) for level in range(2, fmm.plan.nlevels)) < 100_000
    assert fmm.operator.stats()["device_bytes"] < 0.6 * sum(per_offset) * 2 * (p + 1) ** 4 * 8
    out = fmm.evaluate(q)
    phi, grad = O.Fmm(pts, p=p, leaf_points=40).evaluate_helmholtz(k, q)
    errs = [np.linalg.norm(out.potential - phi) / np.linalg.norm(phi),
            np.linalg.norm(out.gradient - grad) / np.linalg.norm(grad)]
    _log(f"  errors {errs}")
    assert max(errs) < tol, errs


def test_host_downloads_of_every_size():
    """Host outputs (through the pinned staging, in chunks of both halves, and the small ones
    past it) against the same evaluation's device outputs, from two threads at once."""
    import threading

    import torch

    _log("case host downloads")
    rng = O.Rng(57)

    def one(n, out):
        pts = rng_pts[n]
        fmm = fmm_amd.FmmBuilder(3).max_points_per_leaf(64).build(pts)
        q = np.cos(np.arange(n))
        host = fmm.evaluate(q)
        phi = torch.empty(n, dtype=torch.float64, device="cuda")
        grad = torch.empty(n, 3, dtype=torch.float64, device="cuda")
        fmm.operator.read_output_device(phi, grad)
        out[n] = np.array_equal(host.potential, phi.cpu().numpy()) and np.array_equal(host.gradient,
                                                                                      grad.cpu().numpy())

    sizes = (2, 700, 2049, 9001, 65_536, 400_003)
    rng_pts = {n: rng.cube(n) for n in sizes}
    out = {}
    work = [threading.Thread(target=lambda part=part: [one(n, out) for n in part]) for part in (sizes[::2], sizes[1::2])]
    for t in work:
        t.start()
    for t in work:
        t.join()
    assert out == {n: True for n in sizes}


def _near_field(plan, q, precision, gradients=True):
    op = fmm_amd.Operator(plan, 3, precision, gradients, 0)
    op.load_charges(q)
    op.reset()
    for level in range(plan.nlevels):
        op.call("p2p", level)
    return op.read_output()


def _near_error(plan, pts, q, out):
    """The largest error of potential and gradient over a bound of the mixed near field.  Each
    f32 operation of a pair's term and of its tile's sum is within 2^-24, and a separation on
    each axis within 2^-28 half-widths from 2^-4.5 on: 1e-6 of the summed magnitudes.  The f64
    positions carry two roundings of 2^-53 of the domain each, 2^(level - 51) half-widths, so both
    of a pair at distance d on three axes move its potential by up to 2^(level - 49) / d of it
    and its force by three times that."""
    leaves, cells = plan.point_leaves().astype(int), plan.leaf_cells()
    counts = np.concatenate([[0], np.cumsum(np.bincount(cells[:, 0], minlength=plan.nlevels))])
    side = plan.domain()[1]
    order = np.argsort(leaves, kind="stable")
    start = np.searchsorted(leaves[order], np.arange(plan.nleaves + 1))
    worst = 0.0
    for level in range(plan.nlevels):
        off, ent = plan.list("near", level)
        half = 0.5 * side / 2.0 ** level
        for r in range(len(off) - 1):
            leaf = counts[level] + r
            t = order[start[leaf]:start[leaf + 1]]
            s = np.concatenate([order[start[e]:start[e + 1]] for e in ent[off[r]:off[r + 1]]])
            d = (pts[t][:, None] - pts[s][None]) / half
            r2 = (d * d).sum(-1)
            with np.errstate(divide="ignore"):
                inv = np.where(r2 == 0, 0.0, 1 / np.sqrt(r2))
            tol = 1e-6 + 2.0 ** (level - 49) * inv
            terms = q[s] * inv
            e = np.abs(out.potential[t] * (4 * np.pi * half) - terms.sum(1)) / ((np.abs(terms) * tol).sum(1) + 1e-60)
            worst = max(worst, e.max(initial=0.0))
            if out.gradient is None:
                continue
            force = -(q[s] * inv**3)[..., None] * d
            size = (np.sqrt((force * force).sum(-1)) * 3 * tol).sum(1) + 1e-60
            g = np.abs(out.gradient[t] * (4 * np.pi * half**2) - force.sum(1)).max(-1) / size
            worst = max(worst, g.max(initial=0.0))
    return worst


@pytest.mark.parametrize("gradients", [True, False])
@pytest.mark.parametrize("leaf,scale", [(2, 1.0), (9, 1e-25), (32, 1.0), (43, 1.0), (70, 1.0)])
def test_mixed_near_field_of_close_pairs(leaf, scale, gradients):
    """The mixed near field alone (fixed-point separations, close pairs from f64) at chunks
    below and above the uniform form's threshold: coincident points, pairs 1e-2 to 1e-12 apart
    inside a leaf and across the faces of boxes."""
    _log(f"case mixed close pairs leaf={leaf} scale={scale} gradients={gradients}")
    rng = O.Rng(63)
    base = rng.cube(2400)
    gaps = 10.0 ** -np.linspace(2, 12, 300)[:, None]
    faces = np.round(rng.cube(200) * 8) / 8 * 0.998 + 0.001
    pts = np.vstack([base, base[:100], base[300:600] + gaps * (rng.cube(300) - 0.5), faces,
                     faces + 1e-9 * (rng.cube(200) - 0.5), [[0.0, 0.0, 0.0], [1.0, 1.0, 1.0]]])
    pts = np.clip(pts, 0.0, 1.0)
    q = rng.normals(len(pts)) * scale
    plan = fmm_amd.Plan(pts, leaf_points=leaf)
    worst = _near_error(plan, pts, q, _near_field(plan, q, "mixed", gradients))
    _log(f"  worst error over its bound {worst:.2f}")
    assert worst < 1.0


def _eight_half_widths_apart(coarse, fine, mirror):
    """Points whose first two are 8 half-widths of the finer one's leaf apart in x, each at the
    outer face of its leaf to 2^-36 of the domain: A in a leaf of `coarse` points, B in one half
    its size with `fine` points, two cells further."""
    corners = np.array([[0.0, 0.0, 0.0], [1.0, 1.0, 1.0]])
    box, side = fmm_amd.Plan(corners, leaf_points=1).domain()
    rng = O.Rng(64)
    a = np.vstack([[0.25 + 2.0**-36, 0.3, 0.3], 0.26 + 0.22 * rng.cube(coarse - 1)])
    b = np.vstack([[0.75 - 2.0**-36, 0.3, 0.3], [0.63, 0.26, 0.26] + 0.11 * rng.cube(fine - 1)])
    rest = [0.51, 0.26, 0.26] + 0.22 * rng.cube(400)
    rest = rest[~((rest[:, 0] > 0.62) & (rest[:, 1] < 0.38) & (rest[:, 2] < 0.38))]
    pts = np.vstack([box[:3] + side * np.vstack([a[:1], b[:1], a[1:], b[1:], rest]), corners])
    if mirror:
        pts[:, 0] = (box[0] + box[3]) - pts[:, 0]
    return pts


@pytest.mark.parametrize("mirror", [False, True])
@pytest.mark.parametrize("coarse,fine", [(3, 4), (30, 30), (50, 50), (3, 50), (50, 4)])
def test_mixed_near_field_at_eight_half_widths(coarse, fine, mirror):
    """The largest separation of a near pair, 8 half-widths (W and X entries moved to the near
    rows, both points on the outer faces of their leaves), is one unit past an int32 in the
    fixed point: the force of the pair alone, in both forms and both directions."""
    _log(f"case mixed eight half-widths coarse={coarse} fine={fine} mirror={mirror}")
    pts = _eight_half_widths_apart(coarse, fine, mirror)
    plan = fmm_amd.Plan(pts, leaf_points=64, near_rule=(300, 300))
    leaves, cells = plan.point_leaves().astype(int), plan.leaf_cells().astype(int)
    u, order = plan.leaf_coordinates()
    at = np.argsort(order)
    la, lb = leaves[0], leaves[1]
    assert cells[la][0] + 1 == cells[lb][0]
    assert (leaves == la).sum() == coarse and (leaves == lb).sum() == fine
    assert abs(u[at[0], 0] - u[at[1], 0]) == pytest.approx(2.0, abs=2.0**-28)
    for source, target in ((0, 1), (1, 0)):
        q = np.zeros(len(pts))
        q[source] = 1.0
        mixed, f64 = _near_field(plan, q, "mixed"), _near_field(plan, q, "f64")
        assert f64.potential[target] > 0  # a near pair
        assert abs(mixed.potential[target] / f64.potential[target] - 1) < 1e-6
        size = np.linalg.norm(f64.gradient[target])
        assert np.abs(mixed.gradient[target] - f64.gradient[target]).max() < 1e-6 * size


@pytest.mark.parametrize("leaf", [1, 9, 20, 42])
@pytest.mark.parametrize("scale,gradients", [(1e30, True), (1e-34, True), (1e30, False), (1e-34, False)])
def test_mixed_near_field_charge_range(leaf, scale, gradients):
    """The staged form over the f32 range of the charges (and of q / r^3 in leaf units)."""
    _log(f"case mixed charge range leaf={leaf} scale={scale} gradients={gradients}")
    rng = O.Rng(65)
    pts = (np.stack(np.meshgrid(*[np.arange(12.0)] * 3), -1).reshape(-1, 3) + 0.5 * rng.cube(12**3)) / 12
    q = rng.normals(len(pts)) * scale
    plan = fmm_amd.Plan(pts, leaf_points=leaf)
    worst = _near_error(plan, pts, q, _near_field(plan, q, "mixed", gradients))
    _log(f"  worst error over its bound {worst:.2f}")
    assert worst < 1.0
