"""The trainer's network kernels at the edges of their 32-row tiles, and with
more tiles than the card has CUs: loss and gradient against the FP64 oracle, and
minibatches against the whole data set."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO
from tests.test_gpu_mlp_train import params_for, small_frames, trainer_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_frames,n", [(1, 2), (1, 31), (1, 32), (1, 33), (3, 21), (70, 121)])
def test_tile_edges(n_frames, n):
    pos, boxes = small_frames(n_frames, n, box=max(1.8, (n / 11.0) ** (1.0 / 3.0)), seed=n)
    # parameters and normalisation of a 64-atom set (two atoms have no spread to normalise by)
    p = params_for(*small_frames())
    rng = np.random.default_rng(n)
    er = rng.normal(-1.0, 0.5, pos.shape[:2])
    fr = rng.normal(0.0, 3.0, pos.shape)
    t = trainer_for(pos, boxes, er, fr, p)
    out, g = t.loss(0.7, 0.05, batch_frames=n_frames, grad=True)
    frames = list(zip(pos, boxes, er, fr))
    ref = MO.loss(p, frames, 0.7, 0.05)
    assert abs(out[0] - ref) <= 1e-4 * ref
    if n_frames <= 3:
        gr = MO.loss_grad(p, frames, 0.7, 0.05)
        gref = np.concatenate([gr[k].ravel() for k in MO.Params.NAMES])
        assert np.linalg.norm(g - gref) <= 2e-3 * np.linalg.norm(gref)
    # minibatches add up to the whole: FP32 sums of the same terms in another order
    _, g2 = t.loss(0.7, 0.05, batch_frames=max(1, n_frames // 3), grad=True)
    assert np.linalg.norm(g2 - g) <= 1e-5 * np.linalg.norm(g)
    t.close()
