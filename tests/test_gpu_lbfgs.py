"""The baseline's L-BFGS direction in two kernels (up to 32 pairs and 32,768 entries)
and as single vector operations beyond, against the oracle."""
import pytest

from diffphd_amd import scenes
from helpers import oracle_body, product_body, rel_err, rollout
from test_oracle_baseline import BASELINE_OPT

pytestmark = pytest.mark.gpu


# Two pairs; 32, the most the kernels take; 33, beyond them once a frame runs longer, which
# the iteration count shows. 81 and 270 entries are at most one for each of the kernels'
# 1,024 threads; 1,512 leave the second turn of their loops ragged. Plain L-BFGS converges to
# rel_tol whatever the history, so the results agree to a small multiple of it (1e-9, as
# for the default history).
@pytest.mark.parametrize("history", [2, 32, 33])
@pytest.mark.parametrize("cells", [(2, 2, 2), (5, 4, 2), (8, 7, 6)])
def test_lbfgs_history_sizes_match_oracle(cells, history):
    spec = scenes.actuated_cantilever(cells=cells)
    opt = dict(BASELINE_OPT, rel_tol=1e-12, abs_tol=1e-12, max_pd_iter=20000, bfgs_history_size=history)
    body = product_body(spec)
    qp, _, _ = rollout(body, spec, 2, opt, method="pd_eigen_pcg")
    qo, _, _ = rollout(oracle_body(spec), spec, 2, opt, method="pd_eigen_pcg")
    print(cells, history, body.last_baseline_stats, rel_err(qp[-1], qo[-1]))
    assert body.last_baseline_stats["pd_iters"] > history + 1
    assert rel_err(qp[-1], qo[-1]) < 1e-9


# 32,760 and 32,775 entries: the last bodies of 3 n entries below and above the switch that
# these grids give; both have more vertices than take the explicit inverse.
@pytest.mark.parametrize("cells,entries", [((20, 19, 25), 32760), ((18, 22, 24), 32775)])
def test_lbfgs_around_the_largest_kernel_form(cells, entries):
    spec = scenes.actuated_cantilever(cells=cells)
    opt = dict(BASELINE_OPT, rel_tol=1e-12, abs_tol=1e-12, max_pd_iter=20000)
    body = product_body(spec)
    assert body.dofs() == entries
    qp, _, _ = rollout(body, spec, 1, opt, method="pd_eigen_pcg")
    qo, _, _ = rollout(oracle_body(spec), spec, 1, opt, method="pd_eigen_pcg")
    print(cells, body.last_baseline_stats, rel_err(qp[-1], qo[-1]))
    assert body.last_baseline_stats["pd_iters"] > 11
    assert rel_err(qp[-1], qo[-1]) < 1e-9
