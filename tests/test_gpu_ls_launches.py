"""Local-search launches at their edges: every size of workgroup the launch rule
takes (test_host_streams.LARGE, where the sizes themselves are checked), and
ADAM steps on both sides of the end of its table of bias corrections."""
import numpy as np
import pytest

import helpers
import oracle as O
from adgpu import search_params
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
