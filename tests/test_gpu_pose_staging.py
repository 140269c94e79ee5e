"""Pose calls in parts: batches around the sizes at which eval_poses and
rescore_f64 go from one staged part to several (8192 poses, then 4096 a part)
give bit for bit what the same poses give in small calls; gradient rows are
written whole; contexts may be called from several threads."""
import ctypes as C
import threading

import numpy as np
import pytest

import adgpu
import helpers

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def bound(gpu_ctx):
    case = helpers.synthetic_case(16, 3, 21, 22, npts=32)
    mid = gpu_ctx.maps_upload(case.packed, case.size, case.maps.num_map_atypes, case.spacing)
    lid = gpu_ctx.ligand_upload(case.tables, case.ep)
    poses = helpers.poses_for(case, 45000, seed=3)
    poses[:, case.ng:] = np.nan   # columns beyond the ligand's genes are not read
    return case, mid, lid, poses


def _in_slices(call, poses, step=1000):
    got = [call(poses[i:i + step]) for i in range(0, len(poses), step)]
    return [np.concatenate([g[k] for g in got]) for k in range(len(got[0]))]


@pytest.mark.parametrize("n", [1, 8191, 8192, 8193, 12289, 45000])
def test_parts_equal_small_calls(gpu_ctx, bound, n):
    case, mid, lid, poses = bound
    p = poses[:n]
    for mode in (adgpu.EVAL_ENERGY, adgpu.EVAL_ENERGRAD, adgpu.EVAL_GRADIENT):
        whole = gpu_ctx.eval_poses(mid, lid, p, mode)
        small = _in_slices(lambda q: gpu_ctx.eval_poses(mid, lid, q, mode), p)
        assert np.array_equal(whole[0], small[0])
        assert np.array_equal(whole[1], small[1])
        assert np.all(whole[1][:, case.ng:] == 0.0)
    whole = gpu_ctx.rescore_f64(mid, lid, p)
    small = _in_slices(lambda q: gpu_ctx.rescore_f64(mid, lid, q), p)
    assert all(np.array_equal(a, b) for a, b in zip(whole, small))
    e, _ = gpu_ctx.eval_poses(mid, lid, p[-60:], adgpu.EVAL_ENERGY)
    helpers.check_energies(case.orc, np.nan_to_num(p[-60:]), e, edge_share=0.2)


def test_outputs_are_whole_and_optional(gpu_ctx, bound):
    case, mid, lid, poses = bound
    fp = C.POINTER(C.c_float)
    p = np.ascontiguousarray(poses[:9000])
    e = np.full(9000, 7.0, np.float32)
    g = np.full((9000, 64), 7.0, np.float32)

    def call(mode, e, g):
        return gpu_ctx.lib.adgpu_eval_poses(gpu_ctx.h, mid, lid, mode, p.ctypes.data_as(fp), 9000,
                                            None if e is None else e.ctypes.data_as(fp),
                                            None if g is None else g.ctypes.data_as(fp))

    assert call(adgpu.EVAL_ENERGRAD, e, g) == 0
    assert np.all(g[:, case.ng:] == 0.0)
    alone_e, alone_g = np.full(9000, 7.0, np.float32), np.full((9000, 64), 7.0, np.float32)
    assert call(adgpu.EVAL_ENERGRAD, alone_e, None) == 0 and np.array_equal(alone_e, e)
    assert call(adgpu.EVAL_ENERGRAD, None, alone_g) == 0 and np.array_equal(alone_g, g)
    untouched = np.full((9000, 64), 7.0, np.float32)
    assert call(adgpu.EVAL_ENERGY, e, untouched) == 0 and np.all(untouched == 7.0)


def test_calls_from_several_threads(gpu_ctx, bound):
    _, mid, lid, poses = bound
    want = [gpu_ctx.eval_poses(mid, lid, poses[k * 9000:(k + 1) * 9000], adgpu.EVAL_ENERGRAD) for k in range(4)]
    got = [None] * 4

    def one(k):
        for _ in range(3):
            got[k] = gpu_ctx.eval_poses(mid, lid, poses[k * 9000:(k + 1) * 9000], adgpu.EVAL_ENERGRAD)

    threads = [threading.Thread(target=one, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(want, got):
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
