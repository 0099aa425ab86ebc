"""GPU: the 2D operators' own gathers (no prefix tables) against the host executor, which
runs the general bodies on the same plan tables: every operator and geometry at the edges of
the line quarters, 64-column groups, 8 x 8 tiles, item groups and fixed column spans.

Tolerance 1e-5 relative L2: the project's bound against FP64; the host's FP32 prefix tables
are within 3e-6 of it on these sizes."""
import numpy as np
import pytest
import torch

from helpers import angles_with_ties, opts2d, rel_l2

pytestmark = pytest.mark.gpu

OPS = ("A", "AT", "B", "BW", "BT", "BWT")
VOLUME_IN = ("A", "BT", "BWT")
SCANS = {"parallel": 0, "flat": 1, "arc": 2}
# name: W, H, Nu, column pitch in pixels at the isocentre, views
SIZES = {
    "one_pixel": (1, 1, 1, 1.0, 5),
    "one_tile": (8, 8, 11, 1.0, 16),
    "odd": (33, 17, 45, 0.9, 23),
    "column_groups": (40, 65, 129, 0.6, 37),
    "wide_columns": (70, 61, 21, 4.7, 19),  # columns over five pixels and more
    "three_pixel_columns": (50, 50, 40, 1.6, 33),
    "fine_columns": (21, 30, 200, 0.13, 40),  # pixels over eight columns and more
}


def _options(size, scan):
    w, h, nu, cell, _ = SIZES[size]
    d = 1.1
    du = cell * d
    if scan == "arc":
        du = du / 500.0
    shu = 0.3 * du
    return opts2d(w, h, nu, d, 0.9 * d, du, 500.0, 1000.0, SCANS[scan], 0.3, -0.2, shu)


@pytest.mark.parametrize("scan", sorted(SCANS))
@pytest.mark.parametrize("size", sorted(SIZES))
def test_slice_operators_match_host(cuda, size, scan):
    from xrecon_amd import _backend as be

    C = be.native()
    opts = [float(v) for v in _options(size, scan)]
    w, h, nu, _, nview = SIZES[size]
    ang = torch.from_numpy(angles_with_ties(nview) if nview >= 16 else 0.3 + np.arange(nview, dtype=np.float32))
    host, plan = C.HostPlan(opts, ang, True), C.Plan(opts, ang, 0, True)
    s = torch.cuda.current_stream(cuda).cuda_stream
    for nb in (1, 2, 5):
        for k, op in enumerate(OPS):
            gen = torch.Generator().manual_seed(100 * nb + k)
            x = torch.rand((nb, 1, h, w) if op in VOLUME_IN else (nb, 1, nview, nu), generator=gen)
            want = host.execute(k, x)
            got = plan.execute(k, x.to(cuda), s)
            assert got.shape == want.shape and torch.isfinite(got).all()
            assert rel_l2(got.cpu().numpy(), want.numpy()) <= 1e-5, (op, nb)
            for b in range(nb):
                assert torch.equal(got[b:b + 1], plan.execute(k, x[b:b + 1].to(cuda), s)), (op, nb, b)


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_slice_bad_values_stay_local(cuda, bad):
    """A NaN or infinity reaches no output that the host executor keeps finite."""
    from xrecon_amd import _backend as be

    C = be.native()
    opts = [float(v) for v in _options("odd", "flat")]
    w, h, nu, _, nview = SIZES["odd"]
    ang = torch.from_numpy(angles_with_ties(nview))
    host, plan = C.HostPlan(opts, ang, True), C.Plan(opts, ang, 0, True)
    s = torch.cuda.current_stream(cuda).cuda_stream
    for k, op in enumerate(OPS):
        x = torch.ones((1, 1, h, w) if op in VOLUME_IN else (1, 1, nview, nu))
        x.view(-1)[[0, x.numel() // 2 + 3, x.numel() - 1]] = bad
        want, got = host.execute(k, x), plan.execute(k, x.to(cuda), s).cpu()
        fine = torch.isfinite(want)
        assert not fine.all() and torch.isfinite(got[fine]).all(), op


def test_slice_batch_of_plans(cuda):
    """A batch of uneven 2D plans equals the plans' own calls bit for bit."""
    from xrecon_amd import _backend as be

    C = be.native()
    s = torch.cuda.current_stream(cuda).cuda_stream
    sizes, nbs = ("odd", "column_groups", "fine_columns", "one_tile"), (1, 2, 3, 4)
    plans = [C.Plan([float(v) for v in _options(z, "arc")], torch.from_numpy(angles_with_ties(SIZES[z][4])), 0, True)
             for z in sizes]
    batch = C.Batch(plans, list(nbs))
    for k, op in enumerate(OPS):
        xs, outs, want = [], [], []
        for i, z in enumerate(sizes):
            w, h, nu, _, nview = SIZES[z]
            img, sino = (nbs[i], 1, h, w), (nbs[i], 1, nview, nu)
            xs.append(torch.rand(img if op in VOLUME_IN else sino, device=cuda))
            outs.append(torch.full(sino if op in VOLUME_IN else img, float("nan"), device=cuda))
            want.append(plans[i].execute(k, xs[i], s))
        ws = torch.empty(max(1, batch.workspace_bytes(k)), dtype=torch.uint8, device=cuda)
        batch.execute_into(k, xs, outs, ws, s)
        for i in range(len(sizes)):
            assert torch.equal(outs[i], want[i]), (op, sizes[i])
