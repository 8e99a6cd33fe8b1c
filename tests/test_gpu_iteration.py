"""The Anderson step on the device (phd_iter.hip) and the next iteration's part that is
queued before the host has decided on this one: windows from none to the largest, a
restart, and an adjoint iterate scaled to the clip norm after its Anderson step.

Capped iterations are compared, not converged results, which a wrong step would still
reach. Both sides run the same iterations and differ by round-off (1e-16 an iteration),
which the least squares of nearly dependent differences multiply; the gates leave a
factor of 1e6 for it."""
import numpy as np
import pytest

from diffphd_amd import scenes
from helpers import backward_frame, oracle_body, product_body, rel_err, rollout

pytestmark = pytest.mark.gpu

GRADS = (0, 1, 3, 4)  # dl_dq, dl_dv, dl_df_ext, dl_dmat_w


def _swinging(seed):
    """A cantilever whose frame starts with a random velocity field, and a loss gradient."""
    spec = scenes.cantilever(cells=(5, 4, 3), seed=seed)
    rng = np.random.default_rng(seed)
    spec["v0"] = (0.3 + seed) * rng.standard_normal(spec["q0"].size)
    for dof, _ in spec["dirichlet"]:
        spec["v0"][dof] = 0.0
    return spec, rng.standard_normal(spec["q0"].size)


def _adjoint(body, spec, frame, g, opt):
    out = backward_frame(body, spec, *frame, 0, g, 0 * g, opt)
    return [out[k] for k in GRADS], body.last_backward_stats()


@pytest.mark.parametrize("dense", [0, 1])
@pytest.mark.parametrize("window", [0, 1, 5, 6])
def test_windows_match_oracle(window, dense):
    spec, g = _swinging(0)
    opt = dict(spec["options"], aa_window=window, phd_dense_inverse=dense, max_pd_iter=30, rel_tol=0.0, abs_tol=0.0)
    prod, orc = product_body(spec), oracle_body(spec)
    frame = rollout(orc, spec, 1, opt)
    q = rollout(prod, spec, 1, opt)[0]
    a, sa = _adjoint(prod, spec, frame, g, opt)
    b, sb = _adjoint(orc, spec, frame, g, opt)
    errs = [rel_err(x, y) for x, y in zip([q[1]] + a, [frame[0][1]] + b)]
    print(window, dense, errs)
    assert sa["backbone_iters"] == sb["backbone_iters"] == 30
    assert max(errs) < 1e-10


# (seed, window, clip norm): window 1 overshoots |s| = 0.2284 to 0.236 around its 16th
# iteration, so that with this clip norm the combined iterate is scaled three times before
# the 20th; windows 5 and 6 restart (|gamma| >= 10) several times within 40 iterations, from a
# full window first.
CASES = {"rescaled": (1, 1, 0.2325), "restart of 5": (1, 5, 1e6), "restart of 6": (1, 6, 1e6)}


@pytest.mark.parametrize("dense", [0, 1])
@pytest.mark.parametrize("case", list(CASES))
def test_adjoint_restart_and_rescale(case, dense):
    seed, window, clip = CASES[case]
    spec, g = _swinging(seed)
    fopt = dict(spec["options"], aa_window=window, phd_dense_inverse=dense)
    bopt = dict(fopt, max_pd_iter=40, rel_tol=0.0, abs_tol=0.0, alg_phd_bwd_clip_norm=clip)
    orc = oracle_body(spec)
    frame = rollout(orc, spec, 1, fopt)
    a, sa = _adjoint(product_body(spec), spec, frame, g, bopt)
    b, sb = _adjoint(orc, spec, frame, g, bopt)
    errs = [rel_err(x, y) for x, y in zip(a, b)]
    print(case, dense, errs, sa["db_norm"])
    assert sa["clipped"] == sb["clipped"] == 0 and sa["backbone_iters"] == 40
    assert max(errs) < 1e-10
    if case == "rescaled":  # and the scaling is seen 20 iterations later
        free, _ = _adjoint(product_body(spec), spec, frame, g, dict(bopt, alg_phd_bwd_clip_norm=1e6))
        assert rel_err(free[0], a[0]) > 1e-3


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("dense", [0, 1])
@pytest.mark.parametrize("case", list(CASES))
def test_queued_front_changes_nothing(case, dense, precision):
    """Phase timing queues nothing ahead: the same bits and iterations with and without."""
    seed, window, clip = CASES[case]
    spec, g = _swinging(seed)
    opt = dict(spec["options"], aa_window=window, phd_dense_inverse=dense, phd_precision=precision)
    bopt = dict(opt, max_pd_iter=40, rel_tol=0.0, abs_tol=0.0, alg_phd_bwd_clip_norm=clip)
    res = []
    for level in (0, 2):
        body = product_body(spec)
        body.timing_enable(level)
        frame = rollout(body, spec, 1, opt)
        out, stats = _adjoint(body, spec, frame, g, bopt)
        res.append(([frame[0][1]] + out, stats))
    assert res[0][1] == res[1][1]
    for x, y in zip(res[0][0], res[1][0]):
        assert np.array_equal(x, y)
