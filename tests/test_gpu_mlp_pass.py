"""The predictor's one-launch pass at the sizes where its path changes: one
feature tile to eight, inputs that fill no tile, the widths and input counts
just past it (layer by layer), one sample, partial tiles of 16 and more tiles
than workgroups.  Against the FP64 oracle: FP32 sums of up to 128 (layers)
and nb (gradients) products through two layers, held to 2e-5 of the norm."""
import numpy as np
import pytest

from oracle import qtn_oracle as O
from qaintensor import learned as Lrn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nin,width", [(1, 16), (5, 32), (63, 48), (72, 128),
                                       (128, 128), (129, 128), (72, 100),
                                       (80, 144)])
@pytest.mark.parametrize("nb", [1, 15, 16, 33, 4600])
def test_pass_matches_oracle(gpu_ctx, nin, width, nb):
    rng = np.random.default_rng(nin + width + nb)
    p = Lrn.init_params(3, nin, width)
    p[:] += (0.05 * rng.standard_normal(p.size)).astype(np.float32)
    X = rng.random((nin, nb)).astype(np.float32)
    T = rng.random(nb).astype(np.float32)
    m = Lrn.RankMLP(p, nin, width, ctx=gpu_ctx)
    y = m.forward(X)
    loss, g = m.loss_grad(X, T)
    X64, p64 = X.astype(np.float64), p.astype(np.float64)
    # the oracle takes the first 64 features through the logarithm
    y_ref = O.mlp_forward(p64, X64, nin, width)[0]
    l_ref, g_ref = O.mlp_loss_grad(p64, X64, T.astype(np.float64), nin, width)
    assert np.abs(y - y_ref).max() <= 2e-5 * max(1.0, np.abs(y_ref).max())
    assert abs(loss - l_ref) <= 2e-5 * max(l_ref, 1e-3)
    assert np.linalg.norm(g - g_ref) <= 2e-5 * max(1.0,
                                                   np.linalg.norm(g_ref))
    # training takes the minibatches in order: the first loss is that of the
    # first half at the initial parameters
    mb = max(1, nb // 2)
    hist = m.train(X, T, steps=3, minibatch=mb, lr=1e-3)
    l0, _ = O.mlp_loss_grad(p64, X64[:, :mb], T[:mb].astype(np.float64), nin,
                            width)
    assert abs(hist[0] - l0) <= 2e-5 * max(l0, 1e-3)
    assert np.all(np.isfinite(hist)) and np.all(np.isfinite(m.params()))
    m.free()


@pytest.mark.parametrize("nin", [70, 72, 80, 127])
def test_infinite_weight_of_the_last_input(gpu_ctx, nin):
    """Inputs that fill no feature tile: the padding takes no part, so an
    infinite weight gives the infinite output it gives without padding."""
    w = 32
    p = np.abs(Lrn.init_params(5, nin, w)) + np.float32(1e-3)
    p[w * (nin - 1) + 7] = np.inf
    X = (np.random.default_rng(nin).random((nin, 20)) + 0.1).astype(np.float32)
    m = Lrn.RankMLP(p, nin, w, ctx=gpu_ctx)
    with np.errstate(all="ignore"):
        ref = O.mlp_forward(p.astype(np.float64), X.astype(np.float64), nin,
                            w)[0]
    assert np.all(ref == np.inf)
    assert np.all(m.forward(X) == np.inf)
    m.free()


@pytest.mark.parametrize("nb", [8192, 8193, 16400])
def test_forward_of_more_tiles_than_workgroups(gpu_ctx, nb):
    p = Lrn.init_params(4, 72, 128)
    X = np.random.default_rng(nb).random((72, nb)).astype(np.float32)
    m = Lrn.RankMLP(p, 72, 128, ctx=gpu_ctx)
    ref = O.mlp_forward(p.astype(np.float64), X.astype(np.float64), 72, 128)[0]
    assert np.abs(m.forward(X) - ref).max() <= \
        2e-5 * max(1.0, np.abs(ref).max())
    m.free()
