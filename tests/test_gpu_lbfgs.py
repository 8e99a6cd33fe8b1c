"""The baseline's L-BFGS direction in two kernels (up to 32 pairs and 32,768 entries)
and as single vector operations beyond, against the oracle."""
import pytest

from diffphd_amd import scenes
from helpers import oracle_body, product_body, rel_err, rollout
from test_oracle_baseline import BASELINE_OPT

pytestmark = pytest.mark.gpu


# Two pairs; 32, the most the kernels take; 33, beyond them once a frame runs longer. Plain
# L-BFGS converges to rel_tol whatever the history, so the results agree to a small
# multiple of it (1e-9, as for the default history).
@pytest.mark.parametrize("history", [2, 32, 33])
@pytest.mark.parametrize("cells", [(2, 2, 2), (5, 4, 2)])
def test_lbfgs_history_sizes_match_oracle(cells, history):
    spec = scenes.actuated_cantilever(cells=cells)
    opt = dict(BASELINE_OPT, rel_tol=1e-12, abs_tol=1e-12, max_pd_iter=20000, bfgs_history_size=history)
    qp, _, _ = rollout(product_body(spec), spec, 2, opt, method="pd_eigen_pcg")
    qo, _, _ = rollout(oracle_body(spec), spec, 2, opt, method="pd_eigen_pcg")
    print(cells, history, rel_err(qp[-1], qo[-1]))
    assert rel_err(qp[-1], qo[-1]) < 1e-9
