"""Images at the ends of single precision's range."""
import numpy as np
import pytest

from lc2registration_amd import engine as E
from lc2registration_amd import synth
from oracle import oracle as O
from test_gpu_parity import LC2_TOL, _oracle_eval, _pair_for, _random_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ndim,r,dims,budget", [
    (2, 2, (37, 29), 0), (2, 9, (44, 39), 0), (2, 3, (37, 29), 1 << 30),
    (3, 2, (24, 21, 13), 0), (3, 5, (27, 19, 14), 0), (3, 2, (24, 21, 13), 1 << 30)])
def test_static_image_whose_gradient_overflows(ndim, r, dims, budget):
    """A fixed high-resolution image of intensities near 1e19: the squares of its gradient
    exceed single precision, so |Sobel| is infinite at part of the voxels and its column drops
    out of the fit there; the intensities alone explain the ultrasound, as in the oracle."""
    w = _random_pair(dims, tuple(d + 9 for d in dims), r, False, ndim, 11)
    # smooth in x < 1/2 (finite gradients), steps of 2e19 beyond
    f = w.fixed.data.astype(np.float64)
    f[..., dims[0] // 2:] *= 2e19
    f[..., :dims[0] // 2] *= 1e15
    w.fixed.data = f.astype(np.float32)
    eng = E.Engine(0, budget)
    p = _pair_for(eng, w, r=r)
    M = p.pose_to_matrix(w.true_pose)
    print(f"overflowing gradient: {ndim}D, r {r}, grid {dims}, budget {budget}", flush=True)
    with np.errstate(all="ignore"):
        res, _, _, G, wm, mm = _oracle_eval(w, M, r=r, maps=True)
    assert np.isinf(G).any() and np.isfinite(G).any() and (mm > 0).any()
    got = p.eval_batch(M[None])
    gm = p.debug_fetch(E.STAGE_MEASURE, M)
    gm = gm[0] if ndim == 2 else gm
    assert np.array_equal(gm > 0, mm > 0)
    assert np.allclose(gm, mm, rtol=1e-7, atol=1e-9)
    assert abs(got.lc2[0] - res.lc2) < LC2_TOL
    p.close()
    eng.close()


@pytest.mark.parametrize("movi", [True, False])
def test_3d_radius_5_where_the_difference_of_two_voxels_overflows(engine, movi):
    """A moving volume whose neighbouring voxels differ by more than single precision holds,
    sampled at whole voxels: the value there is the voxel itself, whatever its neighbours, as in
    the oracle; mutual information is the same with its warped image kept and not (a budget)."""
    r, dims = 5, (24, 21, 15)
    w = _random_pair(dims, dims, r, movi, 3, 12, 1.0)
    rng = np.random.default_rng(3)
    big = rng.random(dims[::-1]) < 0.02 if movi else np.zeros(dims[::-1], bool)
    if movi:
        w.moving.data = np.where(big, 3e38, -1e38 * w.moving.data.astype(np.float64)).astype(np.float32)
    else:  # positive but for the last column, which no patch holds
        w.moving.data = (3e38 * (w.moving.data.astype(np.float64) + 40) / 300).astype(np.float32)
        w.moving.data[..., -1] = -3e38
    w.moving.origin = (0.0, 0.0, 0.0)
    p = _pair_for(engine, w, r=r)
    M = np.eye(3, 4, dtype=np.float32).ravel()
    with np.errstate(all="ignore"):
        res, _, _, _, wm, mm = _oracle_eval(w, M, r=r, maps=True)
    assert (wm > 0).any()
    print(f"overflowing difference: movi {movi}, valid {(wm > 0).sum()}", flush=True)
    got = p.eval_batch(M[None])
    assert np.array_equal(p.debug_fetch(E.STAGE_W, M) > 0, wm > 0)
    assert np.allclose(p.debug_fetch(E.STAGE_MEASURE, M), mm, rtol=1e-7, atol=1e-9 * mm.max())
    assert abs(got.lc2[0] - res.lc2) < LC2_TOL
    if movi:  # the same sampler serves the mutual information's kept warp
        budgeted = E.Engine(0, 1 << 30)
        q = _pair_for(budgeted, w, r=r)
        assert np.array_equal(p.eval_mi(M[None]), q.eval_mi(M[None]))
        q.close()
        budgeted.close()
    p.close()
