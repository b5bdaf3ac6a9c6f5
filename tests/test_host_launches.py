"""How the library plans, allocates and launches, without a GPU: the shared library itself with a HIP runtime in front of
it that hands out host memory, runs no kernel and records what it is asked for (tests/fake_hip.cpp).  Every case runs in
a process of its own, so that the stand-in meets nothing else that uses the runtime."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CASES = {}


def case(fn):
    CASES[fn.__name__] = fn
    return fn


def make(capi, n, dim, metric=0, M=4):
    """An index whose rows and vectors are never looked at."""
    nbrs = np.full((n, 32), -1, np.int32)
    nbrs[:, 0] = (np.arange(n) + 1) % n
    return capi.Index(np.ones((n, dim), np.float32), nbrs, np.arange(M, dtype=np.int32), metric)


def call(idx, Q, k, policy):
    q = np.zeros((Q, idx.dim), np.float32)
    ids, dists = np.empty((Q, k), np.int32), np.empty((Q, k), np.float32)
    return idx.search_device(q.ctypes.data, ids.ctypes.data, dists.ctypes.data, Q, k, policy=policy)


@case
def either_policy_may_be_called_on_a_plan_of_the_other(capi, fake):
    # (visited set, beam) beyond the 64 KB that a kernel takes without being asked: a bitmap of all ids, a table of cells
    # in its bucket form, a long beam
    for n, dim, L, kw in ((600000, 64, 64, dict(visited_slots_log2=-1)), (300000, 200, 600, dict(visited_choices=3, visited_slots_log2=16)),
                          (600000, 200, 64, dict(visited_slots_log2=-1)), (600000, 72, 4096, dict(visited_slots_log2=-1)),
                          (20000, 200, 2000, dict(visited_slots_log2=15))):
        for policy in (1, 0):
            idx = make(capi, n, dim)
            idx.prepare(700, L, policy=policy, best_first_in_lds=True, **kw)
            fake.fake_forget()
            for p in (policy, 1 - policy):
                call(idx, 700, 10, p)
            assert max(fake.fake_launch_lds(i) for i in range(fake.fake_launches())) > 65536, (n, L, policy)
            assert fake.fake_launches_beyond_limit() == 0, (n, L, policy)
            idx.close()


@case
def a_plan_of_one_index_stays_valid_after_a_smaller_one_of_another(capi, fake):
    # the same kernel, with more LDS on the larger index: wavefronts with a bitmap of all ids, four wavefronts per query,
    # the long beam with a larger insert buffer, a workgroup per query
    for nodes, dim, L, Q, policy, kw in (((250000, 20000), 200, 64, 1000, 1, {}), ((600000, 200000), 200, 64, 100, 1, {}),
                                         ((9000, 9000), 96, 2000, 20, 1, dict(best_first_buffer=(1024, 768))),
                                         ((600000, 200000), 200, 64, 100, 0, {})):
        pair = []
        for i, n in enumerate(nodes):
            pair.append(make(capi, n, dim))
            pair[-1].prepare(Q, L, policy=policy, **{k: v[i] for k, v in kw.items()})
        fake.fake_forget()
        for idx in pair:
            call(idx, Q, 10, policy)
        lds = [fake.fake_launch_lds(i) for i in range(fake.fake_launches())]
        assert max(lds) > 65536 and fake.fake_launches_beyond_limit() == 0, (nodes, L, policy, lds)
        for idx in pair:
            idx.close()


@case
def a_best_first_launch_on_the_bitmap_takes_no_visited_state_in_global_memory(capi, fake):
    n, dim, Q, L = 250000, 200, 1000, 64
    state = n * Q  # a byte per node and query slot (n is a multiple of 16)
    idx = make(capi, n, dim)
    for refused in (False, True):  # nor does a refusal of it send the policy to the workgroup-per-query kernel
        fake.fake_refuse(state, state + 1 if refused else state)
        idx.prepare(Q, L, policy=1)
        plan = idx.plan_info()
        assert plan.kernel == 1 and plan.visited_form == 1 and plan.query_slots == Q
        assert fake.fake_live_of_size(state) == 0
    call(idx, Q, 10, 1)
    idx.prepare(Q, L, policy=1, best_first_table_log2=-1)  # without the bitmap the state is there
    assert idx.plan_info().kernel == 0  # (refused: the other kernel)
    fake.fake_refuse(0, 0)
    idx.prepare(Q, L, policy=1, best_first_table_log2=-1)
    assert idx.plan_info().kernel == 1 and fake.fake_live_of_size(state) == 1
    idx.close()


@case
def without_memory_for_what_levels_need_the_search_runs_without_them(capi, fake):
    n, dim, Q, L = 60000, 512, 2000, 256
    pitch = (n + 127) // 128 * 64  # bytes of one query's levels
    for at_least, below in ((n * 4, n * 4 + 1), (pitch * Q, 1 << 40), (8, 9)):  # norms; the block of levels; the norms' largest
        idx = make(capi, n, dim)
        fake.fake_refuse(at_least, below)
        if at_least == 8:  # (as large as the word for the hits of a verification, which is there by now)
            assert fake.fake_live_of_size(8) == 1
        idx.prepare(Q, L)
        plan = idx.plan_info()
        assert plan.visited_form != 6 and plan.screening == 2
        call(idx, Q, 10, 0)
        fake.fake_refuse(0, 0)
        idx.prepare(Q, L)
        assert idx.plan_info().visited_form == 6
        call(idx, Q, 10, 0)
        idx.close()


@case
def the_scratch_of_the_levels_goes_back(capi, fake):
    n, dim, Q, L = 60000, 512, 2000, 256
    least = (n + 127) // 128 * 64 * Q
    idx = make(capi, n, dim)
    idx.prepare(Q, L, threads=512)  # (named: no levels; the copy in codes and the counters are there from here on)
    assert idx.plan_info().visited_form != 6

    def hold_levels():
        idx.prepare(Q, L)
        assert idx.plan_info().visited_form == 6
        return fake.fake_live_bytes()

    for q, again in ((Q, dict(threads=512)), (Q, dict(policy=1, best_first_in_lds=True)), (100, {})):  # plans without
        held = hold_levels()
        idx.prepare(q, L, **again)
        assert fake.fake_live_bytes() < held - least, again
    held = hold_levels()
    fake.fake_forget()
    call(idx, Q, 10, 0)
    levels = fake.fake_launch_fn(fake.fake_launches() - 1)
    assert capi.lib().coral_build_end(idx._h) == 0  # the end of a construction, whose searches plan them too
    assert fake.fake_live_bytes() < held - least and idx.plan_info().visited_form != 6
    call(idx, Q, 10, 0)  # the plan that is left is one without
    assert fake.fake_launch_fn(fake.fake_launches() - 1) != levels and fake.fake_launches_beyond_limit() == 0
    hold_levels()
    idx.close()
    assert fake.fake_live_bytes() == 0


@case
def every_plan_has_its_names(capi, fake):
    idx = make(capi, 60000, 512)
    for Q, L, kw, screening, visited in ((2000, 256, {}, "levels", "lds_levels"), (2000, 256, dict(threads=512), "int8", None),
                                         (100, 64, dict(screening=-1), "none", "lds_bitmap"), (100, 64, dict(screening=1), "fp16", None)):
        idx.prepare(Q, L, **kw)
        plan = idx.plan_info().as_dict()
        assert plan["kernel"] == "beam_search_kernel" and plan["screening"] == screening
        assert visited is None or plan["visited_form"] == visited
    idx.close()


@case
def exact_neighbours_of_a_large_batch_keep_their_scratch(capi, fake):
    # a million points, 10 000 queries, k = 100: lists of 8192 entries, and the matrix of the sample
    idx = capi.Index(np.ones((1000000, 8), np.float32), None, None)
    q = np.zeros((10000, 8), np.float32)
    idx.bruteforce(q, 100)
    kept = fake.fake_live_bytes()
    assert kept > 1000000 * 8 * 4 + (256 << 20)
    fake.fake_refuse(1 << 20, 1 << 40)  # the next call allocates nothing of note
    idx.bruteforce(q, 100)
    assert fake.fake_live_bytes() == kept
    idx.close()


@case
def every_best_first_launch_that_is_accepted_has_its_kernel(capi, fake):
    for dim in (4, 64, 68, 128, 132, 256, 260, 512, 516, 1024, 1028, 2048):
        for metric in (0, 1):
            idx = make(capi, 3000, dim, metric)
            for screening in (-1, 0, 1, 2):
                taken = (screening < 1 or (screening == 1 and dim > 128 and metric == 0) or
                         (screening == 2 and 64 < dim <= 512))
                for L in (4, 128, 129, 256, 257, 512, 513, 1024, 1025, 1280, 1281, 2048):
                    for Q in (1, 5000):
                        try:
                            idx.prepare(Q, L, policy=1, screening=screening, best_first_long=-1)
                        except capi.CoralError as e:
                            assert e.code == capi.ERR_ARG and not taken, (dim, metric, screening, L, Q)
                            continue
                        assert taken, (dim, metric, screening, L, Q)
                        fake.fake_forget()
                        call(idx, Q, min(L, 10), 1)
                        assert idx.plan_info().kernel == 1 and fake.fake_launches_beyond_limit() == 0
                        if screening > 0:
                            assert idx.plan_info().screening == screening
            idx.close()


@case
def best_first_screens_heavy_batches_on_small_graphs_too(capi, fake):
    # fewer than 80 nodes per beam entry: only what memory could not deliver in fp32
    for n, dim, metric, L, cases in ((30000, 512, 1, 759, {1: 0, 900: 0, 960: 2, 5000: 2}),
                                     (30000, 200, 1, 500, {2400: 0, 2500: 2}),
                                     (30000, 512, 0, 500, {1: 0, 1700: 0, 1900: 2, 5000: 2}),
                                     (30000, 512, 0, 1000, {5000: 0}),  # ... and enough of a graph to find new rows in
                                     (30000, 264, 0, 500, {5000: 0}),
                                     (30000, 264, 0, 300, {1: 2, 5000: 2})):
        idx = make(capi, n, dim, metric)
        for Q, screening in cases.items():
            idx.prepare(Q, L, policy=1)
            assert idx.plan_info().screening == screening, (n, dim, metric, L, Q)
        idx.close()


@case
def wavefronts_on_wide_rows_are_workgroups_of_their_own(capi, fake):
    for dim, waves, kw in ((512, 4, {}), (516, 1, {}), (2048, 1, {}), (2048, 4, dict(workgroups=300))):
        idx = make(capi, 9000, dim)
        idx.prepare(1100, 64, policy=1, **kw)
        plan = idx.plan_info()
        assert plan.kernel == 1 and plan.query_slots == 1100
        assert plan.threads == 64 * waves and plan.workgroups == 1100 // waves
        fake.fake_forget()
        call(idx, 1100, 10, 1)
        last = fake.fake_launches() - 1
        assert fake.fake_launch_threads(last) == 64 * waves and fake.fake_launch_blocks(last) == 1100 // waves
        assert fake.fake_launch_lds(last) == plan.lds_bytes
        idx.close()


@case
def batches_of_wide_rows_that_fill_the_caches_take_fewer_at_a_time(capi, fake):
    def kernel(idx, Q):
        idx.prepare(Q, 64, policy=1)
        fake.fake_forget()
        call(idx, Q, 10, 1)
        return fake.fake_launch_fn(fake.fake_launches() - 1)

    for dim, few, many, same in ((2048, 800, 900, False), (1028, 1600, 1700, False), (1024, 1000, 1100, False),
                                 (516, 1800, 2040, True), (512, 1000, 2040, True)):
        idx = make(capi, 9000, dim)
        assert (kernel(idx, few) == kernel(idx, many)) == same, dim
        idx.close()


@case
def full_batches_of_narrow_rows_go_without_the_table(capi, fake):
    for dim, table in ((200, 0), (240, 0), (244, 13)):
        idx = make(capi, 200000, dim)
        idx.prepare(5000, 330, policy=1)
        assert idx.plan_info().visited_slots_log2 == table, dim
        idx.prepare(2048, 330, policy=1)
        assert idx.plan_info().visited_slots_log2 == 13, dim
        idx.close()


@pytest.fixture(scope="module")
def fake_runtime(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fake") / "libfakehip.so")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-Wall", "-D__HIP_PLATFORM_AMD__",
                        "-I/opt/rocm/include", os.path.join(HERE, "fake_hip.cpp"), "-o", out], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return out


@pytest.mark.parametrize("name", sorted(CASES))
def test_host_side(fake_runtime, name):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), fake_runtime, name], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


if __name__ == "__main__":
    sys.path.insert(0, ROOT)
    runtime = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
    for name in ("fake_live_bytes", "fake_live_of_size", "fake_launches", "fake_launch_lds", "fake_launches_beyond_limit"):
        getattr(runtime, name).restype = C.c_size_t
    runtime.fake_live_of_size.argtypes = [C.c_size_t]
    runtime.fake_refuse.argtypes = [C.c_size_t, C.c_size_t]
    runtime.fake_launch_lds.argtypes = runtime.fake_launch_threads.argtypes = runtime.fake_launch_blocks.argtypes = [C.c_size_t]
    runtime.fake_launch_fn.restype, runtime.fake_launch_fn.argtypes = C.c_void_p, [C.c_size_t]
    from coral_amd import capi as binding
    CASES[sys.argv[2]](binding, runtime)
