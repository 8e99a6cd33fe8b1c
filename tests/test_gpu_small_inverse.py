"""The explicit inverse of small bodies (phd_small.hip, option phd_dense_inverse)
against the products with the factor S, over the forms both accept: vertex counts
around the kernels' tile and vector edges, hex and tet, whole-vertex and per-DOF
Dirichlet conditions, contact adjoints, both precisions, and the largest body that
takes it beside the first that does not."""
import numpy as np
import pytest
import torch  # before the library is loaded: both use the same HIP runtime

from diffphd_amd import scenes
from helpers import backward_frame, product_body, rel_err, rollout
from test_oracle_baseline import BASELINE_OPT
from test_oracle_dirichlet import slider

pytestmark = pytest.mark.gpu


def _one_step(spec, opt, seed):
    body = product_body(spec)
    q, v, acts = rollout(body, spec, 1, opt)
    rng = np.random.default_rng(seed)
    out = backward_frame(body, spec, q, v, acts, 0, rng.standard_normal(body.dofs()), np.zeros(body.dofs()), opt)
    return [q[1]] + [out[i] for i in (0, 1, 3, 4)]


def _compare(spec, opt, tol, takes=True):
    """takes: whether the body takes the inverse; where it does not, both are the same bits."""
    a = _one_step(spec, dict(opt, phd_dense_inverse=1), 3)
    b = _one_step(spec, dict(opt, phd_dense_inverse=0), 3)
    errs = [rel_err(x, y) for x, y in zip(a, b)]
    print(spec["name"], spec["V"].shape[1], errs)
    assert max(errs) < tol
    assert all(np.array_equal(x, y) for x, y in zip(a, b)) != takes


# 30 capped iterations from rest: both forms run the same iterations, which carry
# round-off of 1e-16 (FP64) or 6e-8 times the step (mixed) each, and the unconverged
# Anderson iteration multiplies it (by up to 1e2 here); the adjoint's steps
# likewise. 12 to 4,352 vertices: below one 64-row tile, a whole tile (64), one row past
# tiles (385 = 6 x 64 + 1), the switch to four rows per workgroup (990, 1,188), and 4,096 /
# 4,352 around the largest body with an inverse.
@pytest.mark.parametrize("cells", [(2, 1, 1), (3, 3, 3), (4, 6, 10), (7, 6, 5), (10, 9, 8), (11, 10, 8), (15, 15, 15),
                                   (16, 15, 15)])
@pytest.mark.parametrize("precision", [0, 1])
def test_hex_bodies(cells, precision):
    spec = scenes.cantilever(cells=cells, seed=1)
    spec["v0"] = 0.05 * np.random.default_rng(1).standard_normal(spec["q0"].size)
    for dof, _ in spec["dirichlet"]:
        spec["v0"][dof] = 0.0
    opt = dict(spec["options"], max_pd_iter=30, rel_tol=0.0, abs_tol=0.0, phd_precision=precision)
    _compare(spec, opt, 1e-9 if precision == 0 else 1e-4, takes=spec["V"].shape[1] <= 4096)


@pytest.mark.parametrize("precision", [0, 1])
def test_per_dof_dirichlet(precision):
    spec = slider()
    opt = dict(spec["options"], max_pd_iter=30, rel_tol=0.0, abs_tol=0.0, phd_precision=precision)
    _compare(spec, opt, 1e-9 if precision == 0 else 1e-4)


# Vertices and candidates: 168 and 42, 125 and 25 (one row per workgroup); 1,287 and 143,
# 1,331 and 121 (four rows, the last group and every last vector ragged).
@pytest.mark.parametrize("beam_cells,tet_n", [((5, 6, 3), 4), ((12, 10, 8), 10)])
@pytest.mark.parametrize("precision", [0, 1])
def test_contact_adjoint_hex_and_tet(precision, beam_cells, tet_n):
    """Bodies with a boundary keep S in the forward, so q is the same bit for bit; the
    adjoint (backbone and contact-basis correction) takes the inverse."""
    beam = scenes.beam(cells=beam_cells, E=1e5, nu=0.4, seed=2)
    tet = scenes.tet_block(n=tet_n, seed=2)
    tet["v0"] = np.tile([0.0, 0.0, -4.5], tet["V"].shape[1])  # reaches the ground this frame
    for spec in (beam, tet):
        opt = dict(spec["options"], max_pd_iter=12, rel_tol=0.0, abs_tol=0.0, phd_precision=precision,
                   alg_phd_bwd_exact_kpd=1, alg_phd_bwd_kpd_filter=3)
        a = product_body(spec)
        qa, _, acts = rollout(a, spec, 1, opt)
        qb, _, _ = rollout(product_body(spec), spec, 1, dict(opt, phd_dense_inverse=0))
        print(spec["name"], "vertices", a.dofs() // 3, "candidates", len(spec["boundary"][2]))
        assert len(acts[1]) > 0 and np.array_equal(qa[1], qb[1])
        bopt = dict(opt, max_pd_iter=400, rel_tol=1e-12, abs_tol=1e-14)
        g = np.random.default_rng(4).standard_normal(a.dofs())
        res = []
        for dense in (1, 0):
            body = product_body(spec)
            q, v, ac = rollout(body, spec, 1, opt)
            res.append(backward_frame(body, spec, q, v, ac, 0, g, 0 * g, dict(bopt, phd_dense_inverse=dense)))
        errs = [rel_err(res[0][i], res[1][i]) for i in (0, 1, 3, 4)]
        print(spec["name"], "contacts", len(acts[1]), errs)
        assert max(errs) < (1e-8 if precision == 0 else 1e-4)


def _baseline_step(spec, opt, frames):
    body = product_body(spec)
    q, v, acts = rollout(body, spec, frames, opt, method="pd_eigen_pcg")
    g = np.random.default_rng(6).standard_normal(body.dofs())
    out = backward_frame(body, spec, q, v, acts, frames - 1, g, 0 * g, opt, method="pd_eigen_pcg")
    return [q[-1]] + [out[i] for i in (0, 1, 3, 4)], acts[-1]


@pytest.mark.parametrize("scene", ["beam", "napkin"])
def test_baseline_takes_the_option(scene):
    """L-BFGS stops at rel_tol 1e-12 with either form, so results agree to a small
    multiple of it; they are not the same bits, which shows that two forms ran."""
    if scene == "beam":
        spec, frames = scenes.actuated_cantilever(cells=(6, 3, 2)), 1
    else:  # at rest on the sphere: frozen contact nodes, so the columns of A^-1 as well
        spec, frames = scenes.napkin(), 48
    opt = dict(BASELINE_OPT, rel_tol=1e-12, abs_tol=1e-12, max_pd_iter=20000)
    (a, ca), (b, cb) = (_baseline_step(spec, dict(opt, phd_dense_inverse=d), frames) for d in (1, 0))
    errs = [rel_err(x, y) for x, y in zip(a, b)]
    print(scene, "contacts", len(ca), errs)
    assert ca == cb and (scene == "beam" or len(ca) > 0)
    assert max(errs) < 1e-8
    assert not all(np.array_equal(x, y) for x, y in zip(a, b))


def test_baseline_without_the_option_allocates_no_inverse():
    """4,096 vertices: the FP64 inverse is 128 MiB."""
    spec = scenes.actuated_cantilever(cells=(15, 15, 15))
    used = {}
    for dense in (0, 1):
        body = product_body(spec)
        body.factor_build(spec["dt"])
        free = torch.cuda.mem_get_info()[0]
        opt = dict(BASELINE_OPT, rel_tol=0.5, phd_dense_inverse=dense)
        rollout(body, spec, 1, opt, method="pd_eigen_pcg")
        used[dense] = (free - torch.cuda.mem_get_info()[0]) / 2.0**20
    print("MiB", used)
    assert used[0] < 64 and used[1] >= 128
