"""GPU: the voxel gather's slice groups, item pairs and both block paths (every block in the
LDS, or lookups from the table as well): every chunk from 4 slices up and every batch item
give the same bits, and the host executor's results.

Tolerance 1e-5 relative L2: the project's bound against FP64; the host executor is within
2e-7 of it on these operators."""
import numpy as np
import pytest
import torch

from helpers import angles_with_ties, opts3d, rel_l2

pytestmark = pytest.mark.gpu

HALVES = 0x100
OPS = {"AT": 1, "B": 2, "BW": 3}
# W, H, D, Nu, Nv, voxel pitch, slice pitch, column and row pitch at the isocentre, shift z, shift v
SIZES = {
    "tile": (16, 16, 8, 40, 9, 1.0, 1.0, 0.5, 1.0, 0.0, 0.0),
    "odd": (33, 19, 37, 70, 25, 1.0, 1.1, 0.7, 0.9, 0.3, -0.4),
    "tall": (24, 40, 131, 50, 11, 1.0, 0.7, 0.9, 0.8, -5.0, 1.0),  # most slices off the detector
    "one_group": (20, 17, 3, 37, 4, 1.0, 1.0, 0.8, 0.9, 0.0, 0.2),
    "fine_rows": (18, 16, 40, 30, 400, 1.0, 1.0, 0.9, 0.1, 0.0, 0.0),  # blocks beyond the LDS
    "fine_columns": (17, 16, 12, 700, 10, 1.0, 1.0, 0.026, 1.0, 0.0, 0.0),  # rows wider than a block's
    "wide_columns": (48, 48, 20, 9, 12, 1.0, 1.0, 6.3, 1.2, 0.0, 0.0),
}


def _options(size, scan):
    w, h, d, nu, nv, dx, dz, cu, cv, shz, shv = SIZES[size]
    mag = 2.0 if scan == "flat" else 1.0
    du, dv = cu * mag, cv * mag
    if scan == "arc":
        du, dv = cu / 500.0, cv
    sod, sdd = (0.0, 0.0) if scan == "par" else (500.0, 1000.0)
    return opts3d(w, h, d, nu, nv, dx, dx, dz, du, dv, sod, sdd, {"par": 0, "flat": 1, "arc": 2}[scan], 0.3, -0.2, shz,
                  0.2 * du, shv)


@pytest.mark.parametrize("scan", ["par", "flat", "arc"])
@pytest.mark.parametrize("size", sorted(SIZES))
def test_chunks_items_and_block_paths_agree(cuda, size, scan):
    from xrecon_amd import _backend as be

    C = be.native()
    opts = [float(v) for v in _options(size, scan)]
    w, h, d, nu, nv = SIZES[size][:5]
    nview = 70  # more than one run of 64 views
    ang = torch.from_numpy(angles_with_ties(nview))
    host, plan = C.HostPlan(opts, ang, False), C.Plan(opts, ang, 0, False)
    s = torch.cuda.current_stream(cuda).cuda_stream
    for name, op in OPS.items():
        x = torch.rand((3, 1, nview, nv, nu), generator=torch.Generator().manual_seed(op))
        want = host.execute(op, x)
        xd = x.to(cuda)
        ref = plan.execute(op, xd, s)
        assert rel_l2(ref.cpu().numpy(), want.numpy()) <= 1e-5, name
        for nb in (1, 2, 3):
            ws = torch.empty(plan.workspace_bytes(op, nb), dtype=torch.uint8, device=cuda)
            for chunk in (0, 4, 8, 16, 16 | HALVES, 32 | HALVES):
                out = torch.full((nb, 1, d, h, w), float("nan"), device=cuda)
                plan.execute_into(op, xd[:nb].contiguous(), out, ws, s, 0, chunk)
                assert torch.equal(out, ref[:nb]), (name, nb, chunk)


def test_bad_rows_stay_local(cuda):
    """A NaN or infinite sample reaches no voxel that the host executor keeps finite."""
    from xrecon_amd import _backend as be

    C = be.native()
    opts = [float(v) for v in _options("odd", "flat")]
    w, h, d, nu, nv = SIZES["odd"][:5]
    ang = torch.from_numpy(angles_with_ties(20))
    host, plan = C.HostPlan(opts, ang, False), C.Plan(opts, ang, 0, False)
    s = torch.cuda.current_stream(cuda).cuda_stream
    for bad in (float("nan"), float("inf")):
        for name, op in OPS.items():
            x = torch.ones((2, 1, 20, nv, nu))
            x[0, 0, 3, 5, nu // 2] = x[1, 0, 11, nv - 1, nu // 2 + 3] = bad
            want, got = host.execute(op, x), plan.execute(op, x.to(cuda), s).cpu()
            fine = torch.isfinite(want)
            assert not fine.all() and torch.isfinite(got[fine]).all(), name
