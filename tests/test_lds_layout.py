"""The slots of a team's LDS arrays (adgpu_device.h).  On the CPU: for every
kernel shape and every ligand size it takes, each copy of every atom and of the
slot that lanes without an atom write lies inside the array the kernel carves,
and no two of them share a word.  On the GPU: the energy-only kernels with
fewer atoms than a 16-lane team has lanes, where that slot lies nearest to the
team's other data."""
import copy
import os
import shutil
import subprocess
from types import SimpleNamespace

import numpy as np
import pytest

import helpers
import oracle as O
from adgpu import search_params
from adgpu._abi import CLigand

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "adgpu_device.h"
using namespace adgpu;
int main() {
    int bad = 0;
    const int shapes[][2] = {{16, 1}, {16, 2}, {32, 1}, {32, 2}, {32, 4}, {64, 1}, {64, 2}, {64, 4}};
    for (const auto& s : shapes)
        for (int layout = 0; layout < 4; ++layout)
            for (int atoms = 1; atoms <= s[0] * s[1]; ++atoms) {
                const int TW = s[0], NC = s[1];
                const bool PL = layout & 1, GRAD = layout & 2;
                const int words = coord_array(TW, NC, PL, GRAD), stride = slot_stride(atoms);
                std::vector<char> taken(words, 0);
                for (int a = 0; a <= atoms; ++a)
                    for (int c = 0; c < coord_copies(TW, NC, PL, GRAD); ++c) {
                        const int slot = (a < atoms ? a : idle_slot(TW, NC, PL, GRAD, atoms)) + c * stride;
                        if (slot < 0 || slot >= words || taken[slot]) {
                            std::printf("TW %d NC %d PL %d GRAD %d: %d atoms, slot %d of %d words\n", TW, NC, PL, GRAD,
                                        atoms, slot, words);
                            ++bad;
                        } else {
                            taken[slot] = 1;
                        }
                    }
                // room for the coordinates, the forces in gradient kernels, and the genes
                const size_t bytes = 3 * 4 * (size_t)words + (GRAD ? 3 * 4 * (size_t)slot_array(TW, NC) : 0) + 48;
                if (team_bytes_for(TW, NC, 0, PL, GRAD) < bytes) ++bad;
            }
    return bad != 0;
}
"""


def test_every_slot_lies_in_its_array(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    src, exe = str(tmp_path / "slots.hip"), str(tmp_path / "slots")
    with open(src, "w") as f:
        f.write(PROGRAM)
    subprocess.run([hipcc, "-x", "hip", "--cuda-host-only", "-std=c++17", "-w",
                    "-I", os.path.join(REPO, "include"), "-I", os.path.join(REPO, "autodock-gpu_amd", "csrc"),
                    src, "-o", exe], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout[:2000]


@pytest.mark.gpu
@pytest.mark.parametrize("torsions", [0, 1, 3])
@pytest.mark.parametrize("atoms", [9, 13, 14, 15, 16])
def test_narrow_teams_with_idle_lanes(gpu_ctx, atoms, torsions):
    """Initial population, a short Solis-Wets search of it and one generation
    in 16-lane teams: every energy is the oracle's of its pose, with the pairs
    of the whole ligand also where no bond turns.  The search starts at angles
    of 90 to 270 degrees and turns them by a few, so that none is wrapped
    between its evaluation and its storing."""
    case = helpers.synthetic_case(atoms, torsions, 100 * atoms + torsions, 22, npts=40)
    tables = copy.copy(case.tables)
    tables.pairs = np.array([(i, j) for i in range(atoms) for j in range(i + 4, atoms)], np.int32).reshape(-1)
    cl = CLigand(tables)
    case = SimpleNamespace(**{**vars(case), "tables": tables, "cl": cl, "orc": O.Oracle(case.cg, cl, case.ep)})
    mid = gpu_ctx.maps_upload(case.packed, case.size, case.maps.num_map_atypes, case.spacing)
    lid = gpu_ctx.ligand_upload(case.tables, case.ep)
    gpu_ctx.set_team_width(16)
    nrun, pop, job = 3, 50, None
    sp = search_params(num_runs=nrun, pop_size=pop, ls="sw", spacing=case.spacing, max_iters=8)
    sp.base_dang_mul_sqrt3 = 4.0
    init = helpers.poses_for(case, nrun * pop, seed=atoms)
    init[:, 3:case.ng] = np.random.default_rng(atoms).uniform(90, 270, (nrun * pop, case.ng - 3))

    def check():
        d = job.download()
        helpers.check_energies(case.orc, d["pop"], d["ene"], edge_share=0.05)
        return d

    try:
        job = gpu_ctx.job(mid, lid, sp, init, O.cmwc_uints((atoms, torsions), nrun * pop * 64))
        assert job.ls_stats()["team_width"] == 16
        job.initpop()
        first = check()
        job.sum_and_swap()
        job.upload(pop=init, ene=first["ene"])
        job.sum_and_swap()   # the uploaded buffers are those a search works on
        job.kernel_ls()
        job.sum_and_swap()
        searched = check()
        assert np.all(searched["ene"] <= first["ene"]) and np.mean(searched["ene"] < first["ene"]) > 0.5
        job.kernel_gen()
        job.sum_and_swap()
        check()
    finally:
        if job is not None:
            job.destroy()
        gpu_ctx.set_team_width(0)
        gpu_ctx.ligand_release(lid)
        gpu_ctx.maps_release(mid)
