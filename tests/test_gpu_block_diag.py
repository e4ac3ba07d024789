"""The two-level preconditioner's inverse diagonal blocks (meshes that the streamed PCG
solves): fewer steps than the diagonal would take, the same voltages as Jacobi-PCG, on
every lane count and with rows that leave the last tile and its last block partly empty."""
import numpy as np
import pytest

from mpflow_amd.phantom import ellipse_phantom, frame_seed
from tests.problems import eit_of, make_problem, oracle_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rings,L,C,p2,frames,z", [
    (83, 16, 2, False, 2, 0.0),      # 16 lanes, dcFree harmonic
    (84, 32, 2, False, 1, 0.01),     # 64 lanes: electrode unknowns, drive and measurement apart
    (42, 32, 3, True, 2, 0.0),       # P2, 32 lanes
])
def test_block_diagonal_two_level(gpu_ctx, rings, L, C, p2, frames, z):
    import torch
    from mpflow_amd import capi
    from mpflow_amd.eit import SolveOptions
    p = make_problem(rings, L, 1.6 / L, C=C, height=0.4, port_height=0.1, p2=p2)
    if L == 32 and z:
        # measurement pattern independent of the drive: 32 + 32 unique columns
        p["meas"] = np.eye(L) - np.roll(np.eye(L), 3, axis=0)
    eit = eit_of(p, gpu_ctx, frames=frames, contact_impedance=z)
    assert eit.N > 20480
    g = torch.tensor(np.stack([ellipse_phantom(p["nodes"], p["elements"], frame_seed(3, f)) for f in range(frames)]),
                     dtype=torch.float32)
    # refined to 1e-5 * 1e-3 of the right-hand side: both on the FP64 solution to about 1e-8
    kw = dict(stop_rule=capi.MPF_STOP_TOLERANCE, tol=1e-5, precision=capi.MPF_PREC_MIXED, refine_steps=2, refine_tol=1e-3)
    out, steps = {}, {}
    for pre in (0, 1):
        print("case: block diagonal %s preconditioner %d" % ((rings, L, C, p2), pre), flush=True)
        eit.solve(g, SolveOptions(preconditioner=pre, **kw))
        assert eit.last_stats.not_converged == 0
        out[pre], steps[pre] = eit.voltages().cpu().numpy().copy(), eit.last_stats.steps
    err = np.max(np.abs(out[1] - out[0])) / np.max(np.abs(out[0]))
    print("steps", steps, "difference", err)
    assert err < 1e-6
    assert steps[1] < 0.4 * steps[0]
    # warm start, HIP graphs: the same solution again
    eit.solve(g, SolveOptions(preconditioner=1, graphs=1, warm_start=1, **kw))
    again = eit.voltages().cpu().numpy()
    assert np.max(np.abs(again - out[1])) / np.max(np.abs(out[1])) < 1e-6


def _around(p, centers, size):
    """The elements around the nodes nearest to the centres, `size` nodes each (quadratic elements: edge
    nodes, which belong to two elements)."""
    nodes, el = p["nodes"], p["elements"]
    ids = np.unique(el[:, 3:] if el.shape[1] == 6 else el)
    out = np.zeros(el.shape[0], bool)
    for c in centers:
        near = ids[np.argsort(np.linalg.norm(nodes[ids] - c, axis=1))[:size]]
        out |= np.isin(el, near).any(axis=1)
    return out


# (rings, electrodes, harmonics, P2, contact impedance, centres, nodes each): mixed precision must
# converge on the indefinite matrix at all, which the diagonal two-level preconditioner alone decides
@pytest.mark.parametrize("rings,L,C,p2,z,centers,size", [
    (83, 16, 2, False, 0.0, [(0.3, 0.2), (-0.4, 0.1)], 3),         # 16 lanes, dcFree harmonic
    (84, 32, 2, False, 0.01, [(0.3, 0.2), (-0.4, 0.1)], 3),        # 64 lanes, electrode unknowns
    (42, 32, 1, True, 0.0, [(0.3, 0.2)], 1),                       # P2, 32 lanes
])
def test_negative_diagonals_take_the_diagonal(gpu_ctx, rings, L, C, p2, z, centers, size):
    """Linear conductivity may leave a few elements negative after a Gauss-Newton step.  A frame
    with a negative diagonal entry is solved with the signed diagonal, the others beside it with the
    blocks, and both reach the 64-bit solution."""
    import torch
    from mpflow_amd import capi
    from mpflow_amd.eit import SolveOptions
    p = make_problem(rings, L, 1.6 / L, C=C, height=0.4 if C > 1 else 1.0, port_height=0.1 if C > 1 else 1.0, p2=p2)
    if z:
        p["meas"] = np.eye(L) - np.roll(np.eye(L), 3, axis=0)
    eit = eit_of(p, gpu_ctx, frames=3, contact_impedance=z)
    o = oracle_of(p, contact_impedance=z)
    assert eit.N > 20480
    g = np.stack([ellipse_phantom(p["nodes"], p["elements"], frame_seed(5, f)) for f in range(3)]).astype(np.float32)
    g[1, _around(p, centers, size)] = -0.2
    negative = (o.system(g[1].astype(np.float64), 0).diagonal() < 0).sum()
    print("case: negative diagonals %s, %d of them" % ((rings, L, C, p2), negative), flush=True)
    assert negative >= 1
    eit.solve(torch.tensor(g), SolveOptions(stop_rule=capi.MPF_STOP_TOLERANCE, tol=1e-5, precision=capi.MPF_PREC_MIXED,
                                            refine_steps=2, refine_tol=1e-3, preconditioner=1))
    a = eit.voltages().cpu().numpy()
    print("steps", eit.last_stats.steps, "not converged", eit.last_stats.not_converged)
    assert np.isfinite(a).all() and eit.last_stats.not_converged == 0
    for f in range(3):
        # refined to 1e-8 of the right-hand side
        u = o.solve(g[f].astype(np.float64))[0]
        err = np.abs(a[f] - u).max() / np.abs(u).max()
        print("frame %d error %.2e" % (f, err))
        assert err < 1e-6
