"""Local-search launches at their edges: every size of workgroup the launch rule
takes (test_host_streams.LARGE, where the sizes themselves are checked), and
ADAM steps on both sides of the end of its table of bias corrections."""
import numpy as np
import pytest

import helpers
import oracle as O
from adgpu import EVAL_ENERGRAD, search_params, synth
from test_host_streams import LARGE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("atoms, torsions, width, ls, nrun, threads", LARGE)
def test_workgroup_size_leaves_results_alone(gpu_ctx, atoms, torsions, width, ls, nrun, threads):
    """The searches of the first two runs end to the bit as in a job of these
    two alone, which runs in workgroups of 256 threads."""
    case = helpers.synthetic_case(atoms, torsions, lig_seed=atoms, map_seed=4, npts=40)
    mid = gpu_ctx.maps_upload(case.packed, case.size, case.maps.num_map_atypes, case.spacing)
    lid = gpu_ctx.ligand_upload(case.tables, case.ep)
    gpu_ctx.set_team_width(width)
    try:
        pop, got = 150, []
        init = O.initial_population((7,), nrun, pop, case.maps.size_angstr, case.spacing)
        seeds = O.cmwc_uints((7,), nrun * pop * 64)
        for n in (nrun, 2):
            sp = search_params(num_runs=n, pop_size=pop, ls=ls, spacing=case.spacing, max_iters=8)
            job = gpu_ctx.job(mid, lid, sp, init[:n * pop], seeds[:n * pop * 64])
            job.initpop()
            job.kernel_gen()
            job.kernel_ls()
            job.sum_and_swap()
            got.append(job.download())
            job.destroy()
        n = 2 * pop
        assert np.array_equal(got[0]["pop"][:n], got[1]["pop"])
        assert np.array_equal(got[0]["ene"][:n], got[1]["ene"])
        assert np.array_equal(got[0]["evals_runs"][:2], got[1]["evals_runs"])
    finally:
        gpu_ctx.set_team_width(0)
        gpu_ctx.ligand_release(lid)
        gpu_ctx.maps_release(mid)


def _adam_x(g, beta1, beta2, eps, x0, evals, table=None):
    """x of the last pose evaluated in so many ADAM evaluations along a constant
    gradient, in 64 bits; table: the steps whose bias corrections are kept, a
    later step taking the last one's (which is wrong)."""
    b1, b2, eps = float(np.float32(beta1)), float(np.float32(beta2)), float(np.float32(eps))
    x, m, v = x0, 0.0, 0.0
    for t in range(1, evals):
        k = t if table is None else min(t, table)
        m = b1 * m + (1.0 - b1) * g
        v = b2 * v + (1.0 - b2) * g * g
        x -= m / (1.0 - b1 ** k) / (np.sqrt(v / (1.0 - b2 ** k)) + eps)
    return x


@pytest.mark.parametrize("beta1, beta2", [(0.9995, 0.999), (0.0, 0.9995)])
def test_adam_bias_corrections_on_both_sides_of_the_table(gpu_ctx, beta1, beta2):
    """One atom on a map that falls by one unit a grid point along x: the
    gradient is constant, every step lowers the energy, and a step is
    the bias-corrected mean over the root of the corrected square (1) plus an
    epsilon of 19, some 0.05 grid units.  So the position after N evaluations
    tells every correction up to step N - 1, those of the table (1024 steps) and
    those beyond it.  (The atom lies on the axis of every rotation.)

    Bound of the error over n steps: each rounds x below 64 (half an ulp, 2^-19)
    and takes the mean's own error, which the averaging bounds by an ulp over
    1 - beta1, relative (1.2e-4 of a step of 0.05 for beta1 0.9995)."""
    n, evals = 64, (2, 9, 1024, 1025, 1026, 1100)
    x = np.arange(n, dtype=np.float32)
    vals = np.zeros((3, n, n, n), np.float32)
    vals[0] = -x[None, None, :]
    tables = helpers.single_atom_tables(0, 0.0)
    mid = gpu_ctx.maps_upload(synth.pack_maps(vals), (n, n, n), 1, 0.5)
    lid = gpu_ctx.ligand_upload(tables)
    init = np.zeros((2, 64), np.float32)
    init[:, :3] = (2.0, 3.0, 3.0)
    along = np.repeat(init[:1], 4, axis=0)
    along[:, 0] = (2.0, 9.3, 31.7, 56.9)
    _, grad = gpu_ctx.eval_poses(mid, lid, along, EVAL_ENERGRAD)
    # 1023 / 1024: the fixed point rounds halves, and so -1, toward zero
    g = -1023.0 / 1024.0
    assert np.all(grad[:, 0] == g) and not grad[:, 1:3].any()

    def bound(steps):
        return steps * (2.0 ** -19 + (0.05 * 6e-8 / (1.0 - beta1) if beta1 else 0.0))

    got = {}
    for k in evals:
        sp = search_params(num_runs=1, pop_size=2, ls="adam", spacing=0.5, max_iters=k)
        sp.adam_beta1, sp.adam_beta2, sp.adam_epsilon = beta1, beta2, 19.0
        job = gpu_ctx.job(mid, lid, sp, init, O.cmwc_uints((3,), 2 * 64))
        job.initpop()
        job.kernel_gen()   # keeps the better of two equal poses as entity 0
        job.kernel_ls()
        job.sum_and_swap()
        d = job.download()
        job.destroy()
        got[k] = float(d["pop"][0, 0])
        assert abs(got[k] - _adam_x(g, beta1, beta2, 19.0, 2.0, k)) <= bound(k - 1), k
        assert abs(float(d["ene"][0]) + got[k]) <= 1e-4
    gpu_ctx.ligand_release(lid)
    gpu_ctx.maps_release(mid)
    # beyond the table alone, and what a table's last entry in their place would give
    beyond = got[1100] - got[1024]
    want = _adam_x(g, beta1, beta2, 19.0, 2.0, 1100) - _adam_x(g, beta1, beta2, 19.0, 2.0, 1024)
    kept = _adam_x(g, beta1, beta2, 19.0, 2.0, 1100, 1024) - _adam_x(g, beta1, beta2, 19.0, 2.0, 1024, 1024)
    assert abs(beyond - want) <= bound(76)
    assert abs(kept - want) > 3 * bound(76)
