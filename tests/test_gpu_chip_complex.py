"""The on-chip complex conjugate gradients (whole solves in one workgroup per lane group) against
the streamed iteration of the same solve -- a profiled context streams every mesh -- at the edges
of its shapes: one tile, a partial last tile, both lane-group sizes, rows wider than
8 entries, the largest mesh it takes and the first one it does not."""
import numpy as np
import pytest

from tests.problems import make_problem

pytestmark = pytest.mark.gpu

# rings, electrodes, harmonics, P2, frames
SHAPES = [
    (5, 8, 1, False, 1),        # 91 nodes: one tile, one wavefront
    (16, 16, 2, False, 1),      # 817 nodes: four tiles
    (18, 20, 3, False, 1),      # 1027 nodes: one row past 1024, 12 empty lanes
    (14, 16, 2, True, 1),       # P2: rows of 9 and 19 entries
    (20, 16, 3, False, 8),      # 1261 nodes, more groups than CUs
    (36, 16, 1, False, 20),     # two lanes, 3997 nodes
    (51, 16, 1, False, 1),      # 7957 nodes: the largest
    (52, 16, 1, False, 1),      # 8269 nodes: streamed
]


def _solve(eit, g, ctx, streamed, **kw):
    from mpflow_amd import capi
    from mpflow_amd.eit import SolveOptions
    capi.check(capi.lib().mpf_ctx_profile(ctx.h, int(streamed)))
    try:
        eit.solve(g, SolveOptions(**kw))
    finally:
        capi.check(capi.lib().mpf_ctx_profile(ctx.h, 0))
    return eit.voltages(eit.result64).cpu().numpy().copy(), eit.last_stats


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "-".join(map(str, s)))
def test_on_chip_complex_matches_streamed(gpu_ctx, shape):
    import torch
    from mpflow_amd import capi
    from mpflow_amd.eit import EIT
    rings, L, C, p2, frames = shape
    p = make_problem(rings, L, 1.6 / L, C=C, height=1.0 if C == 1 else 0.4, port_height=1.0 if C == 1 else 0.1, p2=p2)
    eit = EIT(p["nodes"], p["elements"], p["boundary"], p["ports"], p["drive"], p["meas"], p["current"], 1.0,
              C, p["height"], p["port_height"], frames=frames, ctx=gpu_ctx, complex_gamma=True)
    rng = np.random.default_rng(7)
    n = (frames, p["elements"].shape[0])
    g = torch.tensor(rng.uniform(0.5, 2.0, n) + 0.3j * rng.uniform(-1.0, 1.0, n), dtype=torch.complex64)
    for herm in (0, 1):
        print("case: on-chip complex %s hermitian %d" % (shape, herm), flush=True)
        # the iteration cap: every pair ends there and says so.  Unconverged voltages are not
        # compared: on the dcFree harmonic the constant mode grows back from rounding after
        # four or five steps, in any summation order
        kw = dict(stop_rule=capi.MPF_STOP_TOLERANCE, tol=1e-12, max_iter=8, complex_hermitian=herm)
        for streamed in (False, True):
            _, st = _solve(eit, g, gpu_ctx, streamed, **kw)
            assert st.max_steps == 8 and st.steps == 8 * C * frames and st.not_converged == C * frames
    # both stop rules to convergence: tol = 1e-6 leaves the FP32 iteration's own error, as the
    # oracle comparison of the same solve allows (2e-5)
    for kw in (dict(stop_rule=capi.MPF_STOP_TOLERANCE, tol=1e-6, max_iter=4000), dict(max_iter=4000)):
        print("case: on-chip complex %s %s" % (shape, kw), flush=True)
        a, sa = _solve(eit, g, gpu_ctx, False, **kw)
        b, sb = _solve(eit, g, gpu_ctx, True, **kw)
        err = np.max(np.abs(a - b)) / np.max(np.abs(b))
        print("steps %d / %d, difference %.2e" % (sa.steps, sb.steps, err))
        assert sa.not_converged == sb.not_converged
        assert err < 4e-5
        assert abs(sa.steps - sb.steps) <= 0.1 * sb.steps + 4


# the same and each lane stride of the sums (rows per pass of the streamed kernels: 64, 32, 16, 8):
# rings, electrodes, harmonics, P2, frames, measurement pattern apart from the drive
ORDER = [
    (5, 8, 1, False, 1, False),       # stride 8: one tile
    (22, 8, 2, False, 3, False),      # stride 8
    (16, 16, 2, False, 3, False),     # stride 16: four tiles
    (20, 16, 3, False, 40, False),    # stride 16, more groups than CUs
    (14, 16, 2, True, 2, False),      # stride 16, rows of 9 and 19 entries
    (18, 20, 3, False, 2, False),     # stride 32, empty lanes
    (30, 32, 1, False, 20, False),    # stride 32, two lanes, two tiles per wavefront
    (29, 16, 1, False, 1, False),     # 11 tiles: the last five wavefronts have one
    (20, 32, 2, False, 2, True),      # stride 64
    (25, 32, 1, True, 2, True),       # stride 64, P2, 30 tiles: 1024 threads
    (30, 32, 1, False, 6, True),      # stride 64, two lanes
    (30, 8, 2, False, 20, False),     # stride 8, two lanes
    (51, 16, 1, False, 2, False),     # 32 tiles: 1024 threads
    (45, 12, 1, False, 1, False),     # 25 tiles: some wavefronts with one tile
    (12, 8, 1, True, 2, False),       # P2, one tile per wavefront: stride 8
    (12, 20, 1, True, 2, False),      # and stride 32
    (30, 8, 1, False, 1, False),      # one lane, two tiles per wavefront: stride 8
    (30, 32, 1, False, 1, False),     # stride 32
    (30, 32, 1, False, 1, True),      # stride 64
    (45, 8, 1, False, 1, False),      # 1024 threads: stride 8
    (45, 24, 1, False, 1, False),     # stride 32
]


@pytest.mark.parametrize("shape", ORDER, ids=lambda s: "-".join(map(str, s)))
def test_on_chip_complex_takes_the_streamed_steps(gpu_ctx, shape):
    """The sums run in the streamed kernels' order: the same steps and the same bits, converged or
    not, and so the streamed solver's error on every input."""
    import torch
    from mpflow_amd import capi
    from mpflow_amd.eit import EIT
    from oracle.eit_oracle import ComplexEITOracle
    rings, L, C, p2, frames, apart = shape
    p = make_problem(rings, L, 1.6 / L, C=C, height=1.0 if C == 1 else 0.4, port_height=1.0 if C == 1 else 0.1, p2=p2)
    if apart:
        p["meas"] = np.eye(L) - np.roll(np.eye(L), 3, axis=0)
    args = (p["nodes"], p["elements"], p["boundary"], p["ports"], p["drive"], p["meas"], p["current"], 1.0, C,
            p["height"], p["port_height"])
    eit = EIT(*args, frames=frames, ctx=gpu_ctx, complex_gamma=True)
    rng = np.random.default_rng(19)
    n = (frames, p["elements"].shape[0])
    for imag in (0.1, 1.0):
        g = torch.tensor(rng.uniform(0.3, 3.0, n) + 1j * imag * rng.uniform(-1.0, 1.0, n), dtype=torch.complex64)
        for kw in (dict(), dict(complex_hermitian=1, max_iter=300), dict(max_iter=9),
                   dict(stop_rule=capi.MPF_STOP_TOLERANCE, tol=1e-6, max_iter=4000)):
            print("case: on-chip complex bits %s imag %g %s" % (shape, imag, kw), flush=True)
            b, sb = _solve(eit, g, gpu_ctx, True, **kw)
            # with no polls the groups give up waiting for the deciding one and go on in the next launch
            for polls in (0, 128):
                capi.check(capi.lib().mpf_ctx_lead_polls(gpu_ctx.h, polls))
                try:
                    a, sa = _solve(eit, g, gpu_ctx, False, **kw)
                finally:
                    capi.check(capi.lib().mpf_ctx_lead_polls(gpu_ctx.h, 128))
                assert (sa.steps, sa.max_steps, sa.not_converged) == (sb.steps, sb.max_steps, sb.not_converged)
                assert np.isfinite(b).all() and np.array_equal(a, b)
    # the last solve (tolerance 1e-6) against the FP64 oracle, with the bound of its own comparison
    if eit.N < 3000:
        u = ComplexEITOracle(*args).solve(g[0].numpy().astype(np.complex128))[0]
        assert np.abs(a[0] - u).max() / np.abs(u).max() < 2e-5
