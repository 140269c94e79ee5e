"""Streams and launches of contexts and jobs, on the CPU: the library's host
code runs on a HIP runtime without a device (fake_hip.cpp), whose streams share
a few modelled hardware queues and whose memory and streams can be bounded."""
import json
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)

PRELUDE = r"""
import ctypes as C, json, sys
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
fake.fake_kernel.restype = C.c_char_p
fake.fake_host_limit.argtypes = fake.fake_allocations_of.argtypes = [C.c_size_t]
sys.path[:0] = [%r, %r, %r]
import numpy as np
import adgpu, helpers
case = helpers.synthetic_case(20, 4, 3, 5, npts=16)

def context():
    ctx = adgpu.Context(0)
    ctx.ids = (ctx.maps_upload(case.packed, case.size, case.maps.num_map_atypes, case.spacing),
               ctx.ligand_upload(case.tables, case.ep))
    return ctx

def job(ctx, nrun=60, ls="fire"):
    sp = adgpu.search_params(num_runs=nrun, pop_size=100, ls=ls, spacing=case.spacing)
    return ctx.job(*ctx.ids, sp, np.zeros((nrun * 100, 64), np.float32), np.ones(nrun * 6400, np.uint32))

def launched(call, kernel):
    fake.fake_clear()
    call()
    return [k for k in range(fake.fake_launches()) if kernel in fake.fake_kernel(k).decode()]

def queues(j):
    "the queue of every run group's local search"
    return [fake.fake_queue(k) for k in launched(lambda: j.run(1), "k_ls_")]

def pose_queue(ctx):
    call = lambda: ctx.eval_poses(*ctx.ids, np.zeros((1, 64), np.float32))
    return fake.fake_queue(launched(call, "k_eval_poses")[0])
""" % (os.path.join(REPO, "autodock-gpu_amd"), os.path.join(REPO, "oracle"), HERE)


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("fake") / "libfakehip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", os.path.join(HERE, "fake_hip.cpp"), "-o", lib],
                   check=True)
    return lib


def run(fake, code, hw_queues=None, **env):
    e = {k: v for k, v in os.environ.items() if not k.startswith("ADGPU_") or k == "ADGPU_LIBRARY"}
    e.pop("GPU_MAX_HW_QUEUES", None)
    if hw_queues:
        e["GPU_MAX_HW_QUEUES"] = str(hw_queues)
    r = subprocess.run([sys.executable, "-c", PRELUDE + code, fake], env=dict(e, **env), capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
    return json.loads(r.stdout.splitlines()[-1])


@pytest.mark.parametrize("hw_queues, groups", [(None, 2), (3, 2), (4, 2), (5, 4), (8, 4)])
@pytest.mark.parametrize("others", [0, 1, 3])
def test_groups_run_apart_and_leave_the_contexts_queue(fake, hw_queues, groups, others):
    """A job's groups have a queue each, and none has that of the context's
    pose calls, however many other contexts took streams before."""
    got = run(fake, """
more = [context() for _ in range(%d)]
ctx = context()
j = job(ctx)
print(json.dumps([queues(j), pose_queue(ctx)]))
""" % others, hw_queues)
    assert len(got[0]) == groups
    assert len(set(got[0] + [got[1]])) == groups + 1, got


def test_jobs_beside_one_that_has_the_lanes(fake):
    """They run in two groups on streams of their own; the lanes go to the next
    job after the first was destroyed."""
    first, second, third = run(fake, """
ctx = context()
a = job(ctx); b = job(ctx)
out = [queues(a), queues(b)]
a.destroy()
c = job(ctx)
print(json.dumps(out + [queues(c)]))
""", 8)
    assert len(second) == 2
    assert len(first) == len(third) == 4 and set(first) == set(third)


def test_lanes_missed_on_a_busy_device_are_looked_for_again(fake):
    """A first job that meets a busy device runs all the same, in as many groups
    as the queues allow; a later one has lanes."""
    first, later = run(fake, """
ctx = context()
fake.fake_busy(1)
a = job(ctx)
fake.fake_busy(0)
out = [queues(a)]
a.destroy()
for _ in range(2):
    b = job(ctx)
    got = queues(b)
    b.destroy()
print(json.dumps(out + [got]))
""", 8)
    assert len(first) == 4
    assert len(later) == 4 and len(set(later)) == 4


def test_a_job_is_not_refused_for_want_of_lanes(fake):
    """Two queues have no four streams apart; the search for them ends where no
    more streams can be had, and gives its own back."""
    got, alive = run(fake, """
fake.fake_streams_limit(6)
ctx = context()
j = job(ctx)
got = queues(j)
j.destroy()
ctx.close()
print(json.dumps([got, fake.fake_streams_alive()]))
""", 2)
    assert len(got) == 2 and alive == 0


@pytest.mark.parametrize("launches", [1, 2, 3, 4, 6, 9])
def test_a_failed_launch_in_the_search_leaves_nothing_running(fake, launches):
    """The search's kernels write to the memory that pose calls use: none may be
    left in flight, whichever launch fails, and the job is not refused."""
    left, groups = run(fake, """
ctx = context()
fake.fake_launches_left(%d)
j = job(ctx, ls="none")
left = fake.fake_unfinished()
fake.fake_launches_left(1 << 30)
print(json.dumps([left, len(launched(lambda: j.run(1), "k_gen"))]))
""" % launches, 8)
    assert left == 0 and groups == 4


def test_searches_for_lanes_become_rare(fake):
    """Where there are no lanes to be found, 32 jobs look for them 6 times."""
    got = run(fake, """
ctx = context()
n = 0
for _ in range(32):
    hold = launched(lambda: job(ctx).destroy(), "k_hold")
    n += bool(hold)
print(json.dumps(n))
""", 1)
    assert got == 6


def test_a_context_opens_without_pinned_memory(fake):
    """Uploads and jobs need no staging memory; a pose call says that it could
    not be had, and asks again the next time."""
    refused, groups, energies = run(fake, """
fake.fake_host_limit(4096)
ctx = context()
try:
    ctx.eval_poses(*ctx.ids, np.zeros((1, 64), np.float32))
    refused = ""
except adgpu.AdgpuError as e:
    refused = str(e)
j = job(ctx)
groups = len(queues(j))
j.destroy()
fake.fake_host_limit(1 << 40)
e, _ = ctx.eval_poses(*ctx.ids, np.zeros((5, 64), np.float32))
print(json.dumps([refused, groups, len(e)]))
""", 4)
    assert "pose staging" in refused and groups == 2 and energies == 5


WORKGROUPS = """
ctx = context()
def threads(atoms, torsions, width, nrun, ls):
    c = helpers.synthetic_case(atoms, torsions, lig_seed=atoms, map_seed=4, npts=16)
    ctx.set_team_width(width)
    ids = ctx.maps_upload(c.packed, c.size, c.maps.num_map_atypes, c.spacing), ctx.ligand_upload(c.tables, c.ep)
    sp = adgpu.search_params(num_runs=nrun, pop_size=150, ls=ls, spacing=c.spacing)
    j = ctx.job(*ids, sp, np.zeros((nrun * 150, 64), np.float32), np.ones(nrun * 9600, np.uint32))
    (k,) = launched(j.kernel_ls, "k_ls_")
    return fake.fake_block(k)
"""


@pytest.mark.parametrize("block, threads", [("64", 64), ("128", 128), ("256", 256), ("512", 256)])
def test_a_fixed_workgroup_size_is_kept(fake, block, threads):
    """Also where launches in workgroups of more threads would hold the pair
    records that 256 threads leave in memory."""
    got = run(fake, WORKGROUPS + """
print(json.dumps([threads(72, 10, 64, 40, ls) for ls in ("sw", "ad", "adam", "fire")]))
""", ADGPU_LS_BLOCK=block)
    assert got == [threads] * 4


# atoms, torsions, team width, local search, runs of 150 searches, and the
# threads of the workgroups that a launch of all their searches takes
LARGE = [(54, 8, 32, "adam", 80, 512), (66, 10, 32, "sw", 80, 512), (80, 12, 32, "adam", 20, 512),
         (80, 12, 32, "fire", 40, 768), (66, 10, 32, "adam", 80, 1024), (80, 12, 32, "sw", 80, 1024),
         (60, 10, 64, "sw", 40, 512), (56, 14, 64, "ad", 80, 512), (64, 10, 64, "ad", 20, 768), (84, 12, 64, "sw", 20, 768),
         (64, 10, 64, "adam", 40, 1024), (84, 12, 64, "fire", 40, 1024), (84, 12, 64, "sw", 40, 1024)]


def test_workgroup_sizes(fake):
    """Larger workgroups than 256 threads are launched where they are meant to
    be: for 32- and 64-lane teams, with and without gradients; two runs of the
    same ligands take 256."""
    got = run(fake, WORKGROUPS + """
print(json.dumps([[threads(*c[:3], n, c[3]) for n in (c[4], 2)] for c in %r]))
""" % (LARGE,))
    assert got == [[c[5], 256] for c in LARGE]


@pytest.mark.parametrize("atoms, width", [(48, 64), (64, 64), (66, 64), (84, 64), (80, 32)])
def test_many_uneven_searches_stay_in_small_workgroups(fake, atoms, width):
    """ADADELTA launches that do not hold all their searches at once, where
    ADAM's take 512 to 1024 threads (56 atoms take 512: LARGE)."""
    ad, adam = run(fake, WORKGROUPS + """
print(json.dumps([threads(%d, 10, %d, 80, ls) for ls in ("ad", "adam")]))
""" % (atoms, width))
    assert ad == 256 and adam >= 512


def test_only_adam_jobs_take_its_table(fake):
    got = run(fake, """
ctx = context()
out = []
for ls in ("sw", "ad", "fire", "adam"):
    fake.fake_clear()
    job(ctx, 3, ls).destroy()
    out.append(fake.fake_allocations_of(8 * 1024))   # 1024 pairs of floats
print(json.dumps(out))
""")
    assert got == [0, 0, 0, 1]
