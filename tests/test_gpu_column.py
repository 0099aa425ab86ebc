"""GPU: the two-step cell gathers (slices of a line summed per detector column, then one
lookup per row boundary) against the host executor, which runs the general z-prefix bodies on
the same plan tables: every operator and geometry at the edges of the row tiles, 64-column
groups, slice pairs and fixed column spans, with lines split over a workgroup and not, and
plans whose rows are too tall for it, which keep the z-prefix gathers.

Tolerance 1e-5 relative L2: the project's bound against FP64; the host executor is within
4e-6 of it on these operators."""
import numpy as np
import pytest
import torch

from helpers import angles_with_ties, opts3d, rel_l2

pytestmark = pytest.mark.gpu

OPS = {"A": 0, "BT": 4, "BWT": 5}
SCANS = {"par": 0, "flat": 1, "arc": 2}
# W, H, D, Nu, Nv, slice pitch, column and row pitch at the isocentre, shift z, shift v, views
SIZES = {
    "one_slice": (9, 8, 1, 11, 1, 1.0, 0.9, 1.0, 0.0, 0.0, 20),
    "one_tile": (24, 20, 17, 64, 16, 1.0, 0.5, 0.9, 0.0, 0.0, 40),
    "tile_and_row": (33, 19, 37, 65, 17, 1.1, 0.7, 0.9, 0.3, -0.4, 40),
    "off_volume": (30, 40, 20, 70, 45, 1.0, 0.7, 0.9, -6.0, 3.0, 40),  # rows above and below the volume
    "unsplit": (24, 20, 9, 129, 33, 1.0, 0.4, 0.5, 0.0, 0.1, 3700),  # more waves than line quarters need
    "tall_rows": (25, 31, 61, 40, 11, 0.5, 0.9, 1.7, 0.2, 0.3, 40),  # tiles of 4 and 8 rows
    "taller_rows": (20, 20, 90, 40, 7, 0.25, 0.9, 2.9, 0.0, 0.0, 40),  # beyond 9 slices per row
    "four_pixels": (50, 50, 12, 21, 10, 1.0, 1.9, 1.0, 0.0, 0.0, 40),
    "wide_columns": (70, 61, 12, 15, 10, 1.0, 4.7, 1.0, 0.0, 0.0, 40),  # columns over five pixels and more
}


def _options(size, scan):
    w, h, d, nu, nv, dz, cu, cv, shz, shv, _ = SIZES[size]
    mag = 2.0 if scan == "flat" else 1.0
    du, dv = cu * mag, cv * mag
    if scan == "arc":
        du, dv = cu / 500.0, cv * 2.0
    sod, sdd = (0.0, 0.0) if scan == "par" else (500.0, 1000.0)
    return [float(v) for v in opts3d(w, h, d, nu, nv, 1.0, 1.1, dz, du, dv, sod, sdd, SCANS[scan], 0.3, -0.2, shz,
                                     0.2 * du, shv)]


def _plans(size, scan):
    from xrecon_amd import _backend as be

    C = be.native()
    opts, ang = _options(size, scan), torch.from_numpy(angles_with_ties(SIZES[size][10]))
    return C, C.HostPlan(opts, ang, False), C.Plan(opts, ang, 0, False)


@pytest.mark.parametrize("scan", sorted(SCANS))
@pytest.mark.parametrize("size", sorted(SIZES))
def test_cell_gathers_match_host(cuda, size, scan):
    C, host, plan = _plans(size, scan)
    w, h, d = SIZES[size][:3]
    s = torch.cuda.current_stream(cuda).cuda_stream
    for name, op in OPS.items():
        x = torch.rand((2, 1, d, h, w), generator=torch.Generator().manual_seed(op))
        want, got = host.execute(op, x), plan.execute(op, x.to(cuda), s)
        assert got.shape == want.shape and torch.isfinite(got).all()
        assert rel_l2(got.cpu().numpy(), want.numpy()) <= 1e-5, name
        for b in range(2):
            assert torch.equal(got[b:b + 1], plan.execute(op, x[b:b + 1].to(cuda), s)), (name, b)


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("size", ["tile_and_row", "four_pixels", "wide_columns"])
def test_bad_values_stay_local(cuda, size, bad):
    """A NaN or infinity reaches no output that the host executor keeps finite."""
    C, host, plan = _plans(size, "flat")
    w, h, d = SIZES[size][:3]
    s = torch.cuda.current_stream(cuda).cuda_stream
    for name, op in OPS.items():
        x = torch.ones((1, 1, d, h, w))
        x[0, 0, d - 2, h // 2, w // 2 + 1] = bad
        want, got = host.execute(op, x), plan.execute(op, x.to(cuda), s).cpu()
        fine = torch.isfinite(want)
        assert not fine.all() and torch.isfinite(got[fine]).all(), name


@pytest.mark.parametrize("scan", sorted(SCANS))
def test_batch_of_plans(cuda, scan):
    """A batch of uneven plans, of every kind of gather, equals the plans' own calls bit for bit."""
    from xrecon_amd import _backend as be

    C = be.native()
    s = torch.cuda.current_stream(cuda).cuda_stream
    sizes, nbs = ("tile_and_row", "unsplit", "taller_rows", "wide_columns", "tall_rows"), (1, 2, 1, 3, 1)
    plans = [C.Plan(_options(z, scan), torch.from_numpy(angles_with_ties(SIZES[z][10])), 0, False) for z in sizes]
    batch = C.Batch(plans, list(nbs))
    for name, op in OPS.items():
        xs, outs, want = [], [], []
        for i, z in enumerate(sizes):
            w, h, d, nu, nv = SIZES[z][:5]
            xs.append(torch.rand((nbs[i], 1, d, h, w), device=cuda))
            outs.append(torch.full((nbs[i], 1, SIZES[z][10], nv, nu), float("nan"), device=cuda))
            want.append(plans[i].execute(op, xs[i], s))
        ws = torch.empty(max(1, batch.workspace_bytes(op)), dtype=torch.uint8, device=cuda)
        batch.execute_into(op, xs, outs, ws, s)
        for i in range(len(sizes)):
            assert torch.equal(outs[i], want[i]), (name, sizes[i])
