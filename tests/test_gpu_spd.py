"""The FP64 factorisation and solve (mpf_spd_solve) at the edges of its 64-row tiles against
numpy's FP64 solve, and a matrix that is not positive definite."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _call(ctx, G, shift, b):
    import torch
    from mpflow_amd import capi
    n = G.shape[0]
    Gd = torch.tensor(G.ravel(order="F"), dtype=torch.float32, device="cuda")
    bd = torch.tensor(b, dtype=torch.float64, device="cuda")
    capi.check(capi.lib().mpf_spd_solve(ctx.h, n, C.c_void_p(Gd.data_ptr()), shift, C.c_void_p(bd.data_ptr()),
                                        C.c_void_p(bd.data_ptr())))
    return bd.cpu().numpy()


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 128, 200, 257, 1024])
def test_spd_solve_tiles(gpu_ctx, n):
    rng = np.random.default_rng(n)
    Q, _ = np.linalg.qr(rng.standard_normal((n, n)))
    G = ((Q * np.logspace(0, -4, n)) @ Q.T).astype(np.float32)
    G = 0.5 * (G + G.T)
    b = rng.standard_normal(n)
    print("case: spd n=%d" % n, flush=True)
    y = _call(gpu_ctx, G, 1e-3, b)          # right-hand side and solution share a buffer
    ref = np.linalg.solve(G.astype(np.float64) + 1e-3 * np.eye(n), b)
    # condition about 1e3: n eps cond is below 1e-9
    assert np.linalg.norm(y - ref) < 1e-9 * np.linalg.norm(ref)


def test_spd_solve_refuses_indefinite(gpu_ctx):
    from mpflow_amd import capi
    G = np.eye(100, dtype=np.float32)
    G[80, 80] = -1.0
    with pytest.raises(capi.MpfError) as e:
        _call(gpu_ctx, G, 0.0, np.ones(100))
    assert e.value.code == capi.MPF_EINVAL
