"""Differential solves of many frames against one Jacobian, which take its products four frames at
a time, against the same frames solved one by one: whole groups of four, remainders, fewer than
four, and rows that do not fill the workgroup."""
import numpy as np
import pytest

from tests.problems import eit_of, make_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rings,electrodes,frames", [(7, 8, 3), (7, 8, 4), (13, 16, 5), (20, 32, 9), (13, 16, 66)])
def test_differential_frames_match_single_frames(gpu_ctx, rings, electrodes, frames):
    import torch
    from mpflow_amd.eit import Solver
    print("case: shared Jacobian", rings, electrodes, frames, flush=True)
    p = make_problem(rings, electrodes, 1.6 / electrodes)

    def solver(n):
        s = Solver(eit_of(p, gpu_ctx, frames=n), 1e-3, gn_refine=4)
        s.pre_solve()
        return s

    one, many = solver(1), solver(frames)
    noise = np.random.default_rng(5).standard_normal((frames,) + tuple(many.measurement.shape[1:]))
    one.eit.solve(torch.ones(1, one.eit.E))
    U = one.eit.result64.cpu().numpy().reshape(1, -1) * (1.0 + 1e-2 * noise)
    many.measurement.copy_(torch.tensor(U, dtype=torch.float64))
    many.solve_differential()
    got = many.material_distribution.cpu().numpy().astype(np.float64)
    for f in range(frames):
        one.measurement.copy_(torch.tensor(U[f:f + 1], dtype=torch.float64))
        one.solve_differential()
        want = one.material_distribution.cpu().numpy().astype(np.float64)[0]
        # FP64 products in another order, refined to 1e-10; the two preparations' FP32 fields,
        # and so their Jacobians, agree to some 1e-6
        assert np.max(np.abs(got[f] - want)) < 1e-5 * np.max(np.abs(want))


@pytest.mark.parametrize("rings,electrodes,frames", [(7, 8, 4), (13, 16, 5), (20, 32, 9)])
def test_differential_frames_match_float64(gpu_ctx, rings, electrodes, frames):
    """The same against the normal equations solved in 64 bits for the model's own Jacobian."""
    import torch
    from mpflow_amd.eit import Solver
    print("case: shared Jacobian in 64 bits", rings, electrodes, frames, flush=True)
    p = make_problem(rings, electrodes, 1.6 / electrodes)
    s = Solver(eit_of(p, gpu_ctx, frames=frames), 1e-3, gn_refine=4)
    s.pre_solve()
    s.eit.solve(torch.ones(frames, s.eit.E), s.options, jacobian=True)
    J = s.eit.jacobian_matrix()[0].cpu().numpy().astype(np.float64)
    U = s.eit.result64[0].cpu().numpy().reshape(-1)
    r = 1e-2 * U * np.random.default_rng(9).standard_normal((frames, U.size))
    s.measurement.copy_(torch.tensor(U + r).reshape(s.measurement.shape))
    s.solve_differential()
    got = s.material_distribution.cpu().numpy().astype(np.float64)
    want = 1.0 + (J.T @ np.linalg.solve(J @ J.T + 1e-6 * np.eye(J.shape[0]), r.T)).T
    err = np.max(np.abs(got - want)) / np.max(np.abs(want))
    print("error %.2e" % err)
    # refined to 1e-10; the result is stored in FP32
    assert err < 1e-6
