"""The on-chip PCG (whole solves in one workgroup per lane group) against the streamed
iteration of the same solve -- a profiled context streams every mesh -- at the edges of its
shapes: one row per thread, a partial last tile, each lane-group size and thread count,
rows wider than 8 entries, the largest mesh it takes and the first one it does not."""
import numpy as np
import pytest

from mpflow_amd.phantom import ellipse_phantom, frame_seed
from tests.problems import eit_of, make_problem, oracle_of

pytestmark = pytest.mark.gpu

# rings, electrodes, harmonics, P2, frames, contact impedance
SHAPES = [
    (5, 8, 1, False, 1, 0.0),       # 91 nodes: one tile, 256 threads
    (16, 16, 1, False, 1, 0.01),    # 833 unknowns: four tiles, one row per thread
    (18, 20, 3, False, 1, 0.0),     # 1027 nodes: one row past 1024, 12 empty lanes
    (14, 16, 2, True, 1, 0.0),      # P2: rows of 9 and 19 entries
    (24, 32, 5, False, 8, 0.0),     # four lanes at 512 threads
    (56, 32, 2, False, 10, 0.0),    # two lanes at 512 threads, 20 rows per thread
    (40, 32, 3, False, 5, 0.01),    # two lanes at 1024 threads
    (82, 16, 1, False, 1, 0.0),     # 20419 nodes: the largest
    (83, 16, 1, False, 1, 0.0),     # 20917 nodes: streamed
]


def _solve(eit, g, ctx, streamed, **kw):
    from mpflow_amd import capi
    from mpflow_amd.eit import SolveOptions
    capi.check(capi.lib().mpf_ctx_profile(ctx.h, int(streamed)))
    try:
        eit.solve(g, SolveOptions(**kw))
    finally:
        capi.check(capi.lib().mpf_ctx_profile(ctx.h, 0))
    return eit.voltages().cpu().numpy().copy(), eit.last_stats


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "-".join(map(str, s)))
def test_on_chip_matches_streamed(gpu_ctx, shape):
    import torch
    from mpflow_amd import capi
    rings, L, C, p2, frames, z = shape
    p = make_problem(rings, L, 1.6 / L, C=C, height=1.0 if C == 1 else 0.4, port_height=1.0 if C == 1 else 0.1, p2=p2)
    eit = eit_of(p, gpu_ctx, frames=frames, contact_impedance=z)
    g = torch.tensor(np.stack([ellipse_phantom(p["nodes"], p["elements"], frame_seed(2, f)) for f in range(frames)]),
                     dtype=torch.float32)
    for pre in (0, 1):
        # FP64 refinement to 1e-5 * 1e-3 of the right-hand side: both land on the FP64
        # solution to about 1e-8 of it, voltages of a condition-limited few times that
        kw = dict(stop_rule=capi.MPF_STOP_TOLERANCE, tol=1e-5, precision=capi.MPF_PREC_MIXED, refine_steps=2,
                  refine_tol=1e-3, preconditioner=pre)
        print("case: on-chip %s preconditioner %d" % (shape, pre), flush=True)
        a, sa = _solve(eit, g, gpu_ctx, False, **kw)
        b, sb = _solve(eit, g, gpu_ctx, True, **kw)
        err = np.max(np.abs(a - b)) / np.max(np.abs(b))
        print("steps %d / %d, difference %.2e" % (sa.steps, sb.steps, err))
        assert sa.not_converged == 0 and sb.not_converged == 0
        assert err < 1e-6
        # the same recurrences in another summation order
        assert abs(sa.steps - sb.steps) <= 0.1 * sb.steps + 4
        # the iteration cap: every pair ends there and says so
        _, sc = _solve(eit, g, gpu_ctx, False, stop_rule=capi.MPF_STOP_TOLERANCE, tol=1e-12, max_iter=5, preconditioner=pre)
        assert sc.max_steps == 5 and sc.steps == 5 * C * frames and sc.not_converged == C * frames
    # the reference rule: column 0 decides for every lane group
    a, sa = _solve(eit, g, gpu_ctx, False)
    b, sb = _solve(eit, g, gpu_ctx, True)
    assert abs(sa.steps - sb.steps) <= 0.1 * sb.steps + 4
    assert np.max(np.abs(a - b)) / np.max(np.abs(b)) < 1e-5


@pytest.mark.parametrize("shape", [SHAPES[1], SHAPES[2], SHAPES[4], SHAPES[5]], ids=lambda s: "-".join(map(str, s)))
def test_groups_that_give_up_waiting_take_the_same_steps(gpu_ctx, shape):
    """Reference rule: with no polls allowed the lane groups stop waiting for the deciding one at once, keep
    their state and go on in the launch after it: the same steps, the same bits."""
    import torch
    from mpflow_amd import capi
    rings, L, C, p2, frames, z = shape
    p = make_problem(rings, L, 1.6 / L, C=C, height=1.0 if C == 1 else 0.4, port_height=1.0 if C == 1 else 0.1, p2=p2)
    eit = eit_of(p, gpu_ctx, frames=frames, contact_impedance=z)
    g = torch.tensor(np.stack([ellipse_phantom(p["nodes"], p["elements"], frame_seed(2, f)) for f in range(frames)]),
                     dtype=torch.float32)
    for kw in (dict(), dict(max_iter=7), dict(preconditioner=1)):
        print("case: on-chip without waiting %s %s" % (shape, kw), flush=True)
        a, sa = _solve(eit, g, gpu_ctx, False, **kw)
        capi.check(capi.lib().mpf_ctx_lead_polls(gpu_ctx.h, 0))
        try:
            b, sb = _solve(eit, g, gpu_ctx, False, **kw)
        finally:
            capi.check(capi.lib().mpf_ctx_lead_polls(gpu_ctx.h, 128))
        assert (sa.steps, sa.max_steps, sa.not_converged) == (sb.steps, sb.max_steps, sb.not_converged)
        assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.parametrize("shape", SHAPES[:7], ids=lambda s: "-".join(map(str, s)))
def test_on_chip_matches_the_oracle(gpu_ctx, shape):
    import torch
    from mpflow_amd import capi
    rings, L, C, p2, frames, z = shape
    p = make_problem(rings, L, 1.6 / L, C=C, height=1.0 if C == 1 else 0.4, port_height=1.0 if C == 1 else 0.1, p2=p2)
    eit, o = eit_of(p, gpu_ctx, frames=frames, contact_impedance=z), oracle_of(p, contact_impedance=z)
    g = np.stack([ellipse_phantom(p["nodes"], p["elements"], frame_seed(2, f)) for f in range(frames)]).astype(np.float32)
    u = np.stack([o.solve(x.astype(np.float64))[0] for x in g])
    # FP64 refinement to 1e-8 of the right-hand side; FP32 to 1e-6 with the iteration's own error, as the
    # forward solves' comparisons allow
    mixed = dict(precision=capi.MPF_PREC_MIXED, tol=1e-5, refine_steps=2, refine_tol=1e-3)
    for pre in (0, 1):
        for kw, bound in ((mixed, 1e-6), (dict(tol=1e-6), 2e-5)):
            print("case: on-chip against the oracle %s preconditioner %d" % (shape, pre), flush=True)
            a, st = _solve(eit, torch.tensor(g), gpu_ctx, False, stop_rule=capi.MPF_STOP_TOLERANCE, preconditioner=pre, **kw)
            err = np.max(np.abs(a - u)) / np.max(np.abs(u))
            print("error %.2e" % err)
            assert st.not_converged == 0 and err < bound
