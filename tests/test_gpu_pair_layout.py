"""The pair loop's padded records: pair counts at and around the team widths
(the last step of the loop, its padding, no pairs at all), other exponents and
CG-G0 bonds, energies and merged gradients against the FP32 oracle with the
bars of test_gpu_parity."""
import copy
from types import SimpleNamespace

import numpy as np
import pytest

import adgpu
import helpers
import oracle as O
from adgpu._abi import CLigand

pytestmark = pytest.mark.gpu


def _with(case, **kw):
    t = copy.copy(case.tables)
    for k, v in kw.items():
        setattr(t, k, v)
    cl = CLigand(t)
    return SimpleNamespace(**{**vars(case), "tables": t, "cl": cl, "orc": O.Oracle(case.cg, cl, case.ep)})


def _forms(c1):
    pairs = np.asarray(c1.tables.pairs).reshape(-1, 2)
    for n in (0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 129):
        yield _with(c1, pairs=pairs[:n].reshape(-1))
    exps = np.array(c1.tables.vw_exp).copy()
    exps[1::3] = (9 << 8) + 7
    yield _with(c1, vw_exp=exps)                     # exponents other than 12-6 / 12-10
    types = np.array(c1.tables.atype_reqm).copy()
    types[:2] = (24, 25)
    yield _with(c1, atype_reqm=types)                # CG-G0 bond terms


@pytest.mark.parametrize("width", [16, 32, 64])
def test_padded_pairs(gpu_ctx, c1, width):
    mid = gpu_ctx.maps_upload(c1.packed, c1.size, c1.maps.num_map_atypes, c1.spacing)
    gpu_ctx.set_team_width(width)
    try:
        for case in _forms(c1):
            lid = gpu_ctx.ligand_upload(case.tables, case.ep)
            poses = helpers.poses_for(case, 120, seed=77)
            e, g = gpu_ctx.eval_poses(mid, lid, poses, adgpu.EVAL_ENERGRAD)
            helpers.check_energies(case.orc, poses, e, edge_share=0.05)
            e2, _ = gpu_ctx.eval_poses(mid, lid, poses, adgpu.EVAL_ENERGY)
            helpers.check_energies(case.orc, poses, e2, e_ref=e, edge_share=0.05)
            well = [0, 1, 2] + list(range(6, case.ng))
            quantum = np.array([helpers.gene_quantum(case, k) for k in range(case.ng)])
            off = 0
            for p, row in zip(poses, g):
                _, go = case.orc.energrad32(p, True)
                off += int((np.abs(row[:case.ng] - go)[well] > (1e-4 * np.abs(go) + 4 * quantum)[well]).sum())
            assert off <= 0.002 * len(poses) * len(well)
            assert np.all(g[:, case.ng:] == 0.0)
            gpu_ctx.ligand_release(lid)
    finally:
        gpu_ctx.set_team_width(0)
        gpu_ctx.maps_release(mid)


@pytest.mark.parametrize("ls", ["adam", "sw"])
@pytest.mark.parametrize("atoms, torsions, width", [(54, 8, 64), (72, 10, 64), (45, 8, 32)])
def test_large_workgroups(gpu_ctx, atoms, torsions, width, ls):
    """Local searches in the workgroups that a launch of many searches takes
    when 256-thread ones could not all hold the pair records: the searches of
    a job of 40 runs end as in a job of the first 2 runs, which fit at once."""
    case = helpers.synthetic_case(atoms, torsions, lig_seed=atoms, map_seed=4, npts=40)
    mid = gpu_ctx.maps_upload(case.packed, case.size, case.maps.num_map_atypes, case.spacing)
    lid = gpu_ctx.ligand_upload(case.tables, case.ep)
    gpu_ctx.set_team_width(width)
    try:
        pop, got = 150, []
        init = O.initial_population((5,), 40, pop, case.maps.size_angstr, case.spacing)
        seeds = O.cmwc_uints((5,), 40 * pop * 64)
        for nrun in (40, 2):
            sp = adgpu.search_params(num_runs=nrun, pop_size=pop, ls=ls, spacing=case.spacing, max_iters=12)
            job = gpu_ctx.job(mid, lid, sp, init[:nrun * pop], seeds[:nrun * pop * 64])
            job.initpop()
            job.generation()
            got.append(job.download())
            job.destroy()
        n = 2 * pop
        assert np.array_equal(got[0]["pop"][:n], got[1]["pop"])
        assert np.array_equal(got[0]["ene"][:n], got[1]["ene"])
        helpers.check_energies(case.orc, got[0]["pop"][::97], got[0]["ene"][::97], edge_share=0.2)
    finally:
        gpu_ctx.set_team_width(0)
        gpu_ctx.ligand_release(lid)
        gpu_ctx.maps_release(mid)


def test_adam_past_its_table(gpu_ctx, c1):
    """ADAM searches around the end of the job's table of bias corrections
    (1024 steps): a longer search keeps the shorter one's steps, so its best
    energy is at most the shorter one's, and is the energy of its pose."""
    mid = gpu_ctx.maps_upload(c1.packed, c1.size, c1.maps.num_map_atypes, c1.spacing)
    lid = gpu_ctx.ligand_upload(c1.tables, c1.ep)
    init = O.initial_population((9,), 1, 16, c1.maps.size_angstr, c1.spacing)
    seeds = O.cmwc_uints((9,), 16 * 64)
    last = None
    for iters in (1023, 1024, 1025, 1100):
        sp = adgpu.search_params(num_runs=1, pop_size=16, ls="adam", spacing=c1.spacing, max_iters=iters)
        job = gpu_ctx.job(mid, lid, sp, init, seeds)
        job.initpop()
        job.kernel_gen()
        job.kernel_ls()
        job.sum_and_swap()
        d = job.download()
        job.destroy()
        # the initial energies, 15 offspring, then one evaluation a step of every searched entity
        assert int(d["evals_runs"][0]) == 16 + 15 + 16 * iters
        helpers.check_energies(c1.orc, d["pop"], d["ene"], edge_share=0.3)
        if last is not None:
            assert np.all(d["ene"] <= last)
        last = d["ene"]
    gpu_ctx.ligand_release(lid)
    gpu_ctx.maps_release(mid)


@pytest.mark.parametrize("atoms, torsions, width", [(65, 8, 64), (66, 8, 32), (90, 12, 64), (130, 12, 64)])
def test_compact_pair_records(gpu_ctx, atoms, torsions, width):
    """Gradient kernels read the pairs of more than 64 atoms in 24 bytes: energies
    and gradients with both exponents, with others and with CG-G0 bonds, whose
    terms the compact record leaves to the flags."""
    case = helpers.synthetic_case(atoms, torsions, lig_seed=atoms, map_seed=4, npts=48)
    exps = np.array(case.tables.vw_exp).copy()
    ten = exps.copy()
    ten[::2] = (12 << 8) + 10
    exps[1::3] = (9 << 8) + 7
    types = np.array(case.tables.atype_reqm).copy()
    types[:2] = (24, 25)
    mid = gpu_ctx.maps_upload(case.packed, case.size, case.maps.num_map_atypes, case.spacing)
    gpu_ctx.set_team_width(width)
    try:
        for form in (case, _with(case, vw_exp=ten), _with(case, vw_exp=exps), _with(case, atype_reqm=types)):
            lid = gpu_ctx.ligand_upload(form.tables, form.ep)
            poses = helpers.poses_for(form, 60, seed=78)
            e, g = gpu_ctx.eval_poses(mid, lid, poses, adgpu.EVAL_ENERGRAD)
            helpers.check_energies(form.orc, poses, e, edge_share=0.05)
            e2, _ = gpu_ctx.eval_poses(mid, lid, poses, adgpu.EVAL_ENERGY)
            helpers.check_energies(form.orc, poses, e2, e_ref=e, edge_share=0.05)
            well = [0, 1, 2] + list(range(6, form.ng))
            quantum = np.array([helpers.gene_quantum(form, k) for k in range(form.ng)])
            off = 0
            for p, row in zip(poses, g):
                _, go = form.orc.energrad32(p, True)
                off += int((np.abs(row[:form.ng] - go)[well] > (1e-4 * np.abs(go) + 4 * quantum)[well]).sum())
            assert off <= 0.002 * len(poses) * len(well)
            gpu_ctx.ligand_release(lid)
    finally:
        gpu_ctx.set_team_width(0)
        gpu_ctx.maps_release(mid)
