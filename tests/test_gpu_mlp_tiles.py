"""The network's matrix products at the edges of their tiles against the FP64 oracle with the
device's BF16 operand rounding: sizes that are no multiple of 4, one row, fewer than 4 columns,
remainders of the 64- and 128-wide tiles and of the K step, products split over K (few rows)
and tiles of 128."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,batch", [
    ([5, 3, 2], 1),                   # everything smaller than one vector
    ([131, 65, 63, 3], 1),            # one row, remainders of every kind
    ([1030, 514, 129], 7),            # 8 and 4 slices of K
    ([512, 1027, 640, 301], 64),      # whole rows, ragged columns, split
    ([70, 2050, 65], 2177),           # tiles of 128 with a remainder on both sides
])
def test_mlp_products_at_tile_edges(gpu_ctx, dims, batch):
    import torch
    from mpflow_amd.learned import Mlp
    from oracle.mlp_oracle import MlpOracle
    print("case: mlp tiles", dims, batch, flush=True)
    net = Mlp(dims, seed=9, ctx=gpu_ctx)
    rng = np.random.default_rng(17)
    X = rng.standard_normal((batch, dims[0])).astype(np.float32)
    T = (0.3 * rng.standard_normal((batch, dims[-1]))).astype(np.float32)
    ora = MlpOracle(dims, net.params())
    Y = net.forward(torch.tensor(X, device="cuda")).cpu().numpy()
    Yo, _ = ora.forward(X, bf16=True)
    loss = net.backward(torch.tensor(T, device="cuda"))
    g = net.params(grads=True)
    lo, go = ora.grads_flat(X, T, bf16=True)
    ey = float(np.linalg.norm(Y - Yo) / np.linalg.norm(Yo))
    eg = float(np.linalg.norm(g - go) / np.linalg.norm(go))
    print("forward %.2e, loss %.6f vs %.6f, grads %.2e" % (ey, loss, lo, eg))
    # the BF16 oracle rounds the same operands; what is left is FP32 accumulation and the
    # activations it moves across a BF16 boundary (2^-8 of a value, one in some hundreds): a
    # wrong or missing term would be 1 / sqrt(K) or more
    assert ey < 2e-3
    assert abs(loss - lo) < 1e-3 * lo
    assert eg < 3e-3


@pytest.mark.parametrize("dims", [[3001, 4099, 33], [33, 4099, 3001], [700, 900, 9]])
def test_mlp_parameters_read_back_as_set(gpu_ctx, dims):
    """Above and below the size that is read by several threads, with ragged last chunks."""
    from mpflow_amd.learned import Mlp
    print("case: mlp read back", dims, flush=True)
    net = Mlp(dims, seed=1, ctx=gpu_ctx)
    w = np.random.default_rng(3).standard_normal(net.n_params).astype(np.float32)
    net.set_params(w)
    for _ in range(2):
        np.testing.assert_array_equal(net.params(), w)
