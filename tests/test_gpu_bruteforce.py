"""Exact brute-force kNN on the GPU (the ground-truth / builder-kNN component that replaces
faiss): bit-exact against the oracle's brute force in the same summation order, and within
tolerance of the fp64 closed form."""
import time

import numpy as np
import pytest

from coral_amd import capi, synth, workloads

pytestmark = pytest.mark.gpu
SEQ = 0  # ORDER_GPU_SEQ


def test_comp_gt_tool_and_vectors_only_index(orc, tmp_path):
    """The ground-truth driver: fbin in, gt file out (layout of tests/comp_gt.cpp:142-175)."""
    import os
    import subprocess
    from coral_amd import formats
    n, dim, Q, k = 6000, 100, 50, 20
    base = synth.gaussian_matrix(5, n, dim)
    q = synth.shifted_queries(Q, dim, 6, 7, 8)
    formats.fbin_write(tmp_path / "base.fbin", base)
    formats.fbin_write(tmp_path / "query.fbin", q)
    tool = os.path.join(os.path.dirname(capi.LIB_PATH), "comp_gt")
    for dist, m in (("l2", capi.L2), ("ip", capi.IP)):
        r = subprocess.run([tool, "--base_data_path", str(tmp_path / "base.fbin"), "--query_data_path",
                            str(tmp_path / "query.fbin"), "--gt_save_file", str(tmp_path / "gt.bin"), "--k", str(k),
                            "--nq", "40", "--dist", dist], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr
        gt = formats.gt_read(tmp_path / "gt.bin")
        assert gt.shape == (40, k)
        b2, q2 = (formats.normalize_l2(base), formats.normalize_l2(q)) if dist == "ip" else (base, q)
        oi, _ = orc.bruteforce(b2, q2[:40], k, m, order=SEQ)
        assert np.array_equal(gt, oi)
    r = subprocess.run([tool, "--dist", "l2"], capture_output=True, text=True)
    assert r.returncode == 255 and "required but missing" in r.stderr
    # a vectors-only index serves brute force and refuses graph search
    idx = capi.Index(base, None, None)
    ids, _, _ = idx.bruteforce(q, k)
    assert np.array_equal(ids, orc.bruteforce(base, q, k, order=SEQ)[0])
    with pytest.raises(capi.CoralError) as e:
        idx.search(q, 5, 16)
    assert e.value.code == capi.ERR_STATE
    idx.close()


def ring(n, R=2):
    g = np.full((n, R), -1, np.int32)
    g[:, 0] = (np.arange(n) + 1) % n
    return g


@pytest.mark.parametrize("n,dim,Q,k,metric,tomb", [
    (3000, 200, 37, 100, "l2", False),
    (3000, 200, 37, 100, "ip", False),
    (5000, 20, 130, 10, "l2", True),
    (777, 132, 5, 129, "l2", False),
    (4097, 4, 257, 1, "ip", True),
    (50, 8, 9, 64, "l2", True),      # fewer live points than k: padded
    (20000, 128, 300, 32, "l2", False),
])
def test_bruteforce_exact_against_oracle(orc, n, dim, Q, k, metric, tomb):
    m = capi.IP if metric == "ip" else capi.L2
    base = synth.gaussian_matrix(n + dim, n, dim)
    q = synth.shifted_queries(Q, dim, 3, 4, 5)
    if metric == "ip":
        base, q = synth.normalize_rows(base), synth.normalize_rows(q)
    mask = synth.tombstone_mask(n, 77, 3) if tomb else None
    idx = capi.Index(base, ring(n), np.array([0], np.int32), m)
    if tomb:
        idx.set_deleted(mask)
    ids, dists, _ = idx.bruteforce(q, k, have_delete=tomb)  # matrix-core screening + exact re-ranking
    redone, fused = idx.bruteforce_last_redone(), idx.bruteforce_last_fused()
    idx.bruteforce_exact_only(2)                            # the screening's candidates from the distance matrix
    ids3, dists3, _ = idx.bruteforce(q, k, have_delete=tomb)
    assert idx.bruteforce_last_fused() == 0 and idx.bruteforce_last_redone() == redone
    assert np.array_equal(ids3, ids) and dists3.tobytes() == dists.tobytes()
    idx.bruteforce_exact_only(True)                         # every pair in the reference's order
    ids2, dists2, _ = idx.bruteforce(q, k, have_delete=tomb)
    assert idx.bruteforce_last_redone() == 0 and idx.bruteforce_last_fused() == 0
    idx.close()
    assert fused == (1 if n >= 8192 else 0)  # 64 tiles of 128 points are what the sample needs
    print("queries that the screening could not vouch for: %d of %d" % (redone, Q), flush=True)
    oi, od = orc.bruteforce(base, q, k, m, deleted=mask, order=SEQ)
    assert np.array_equal(ids, oi)
    assert dists.tobytes() == od.tobytes()
    assert np.array_equal(ids2, oi) and dists2.tobytes() == od.tobytes()
    if n > 2 * (k + 32) and dim >= 20:
        assert redone <= Q // 4  # independent data: the candidates nearly always suffice
    # against the fp64 closed form: same ids except where fp32 rounding reorders near-ties
    ti, td = orc.bruteforce(base, q, k, m, deleted=mask)
    live = ti >= 0
    assert (ids[live] == ti[live]).mean() > 0.98
    assert np.allclose(dists[live], td[live], rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("n,dim,Q,k,metric,law", [
    (8192, 4, 1, 1, "l2", "plain"),            # one query in a tile of 256, a quarter of one stage of 16 dimensions
    (8319, 12, 255, 10, "ip", "plain"),        # last base tile one short, last query tile one short
    (8321, 16, 256, 10, "l2", "plain"),        # last base tile of one point; whole tile of queries, whole stage
    (9000, 20, 257, 33, "ip", "plain"),        # a second query tile of one
    (20483, 36, 1025, 10, "l2", "plain"),      # two passes over the base with a tightened bound
    (20483, 24, 1024, 100, "ip", "plain"),
    (9000, 24, 40, 128, "l2", "plain"),        # 160 kept candidates: the last that 256 threads select
    (9000, 24, 40, 129, "l2", "plain"),
    (9000, 24, 4097, 5, "ip", "plain"),        # a second block of queries, of one
    (9000, 24, 2049, 5, "l2", "plain"),        # a second piece of the sample, of one
    (20483, 24, 4097, 5, "l2", "plain"),       # both, in two passes over the base
    (20483, 24, 2049, 5, "ip", "plain"),
    (20483, 24, 1024, 10, "l2", "spread"),     # rows from 0.1 to 10 in one base, each on a scale of its own
    (20483, 24, 300, 10, "ip", "spread"),
    (20483, 24, 1024, 10, "l2", "row_scales"),  # rows from 1e-12 to 1e12: nothing can be vouched for
    (20483, 24, 300, 10, "ip", "row_scales"),
    (8500, 24, 130, 10, "l2", "tiny"),         # squared norms at the end of the range: scales are clamped
    (8500, 24, 130, 10, "ip", "tiny"),
    (8500, 24, 40, 10, "ip", "huge_row"),      # a squared norm that overflows: nothing can be vouched for
])
def test_screening_on_split_halves_at_the_edges_of_its_tiles(orc, n, dim, Q, k, metric, law):
    """Sizes around the tiles (256 queries, 128 points, 16 dimensions) and magnitudes around the ends of the scaling;
    the result is defined bit for bit, so there is nothing to tolerate."""
    m = capi.IP if metric == "ip" else capi.L2
    base = synth.gaussian_matrix(n + 3 * dim, n, dim)
    q = synth.shifted_queries(Q, dim, 13, 14, 15)
    rs = np.random.RandomState(n)
    if law == "row_scales":
        base *= (10.0 ** rs.uniform(-12, 12, (n, 1))).astype(np.float32)
    elif law == "spread":
        base *= (10.0 ** rs.uniform(-1, 1, (n, 1))).astype(np.float32)
    elif law == "tiny":
        base *= np.float32(1e-19)
        q *= np.float32(1e-19)
    elif law == "huge_row":
        base[n // 2] *= np.float32(1e20)
    idx = capi.Index(base, None, None, m)
    ids, dists, _ = idx.bruteforce(q, k)
    redone, fused = idx.bruteforce_last_redone(), idx.bruteforce_last_fused()
    idx.close()
    oi, od = orc.bruteforce(base, q, k, m, order=SEQ)
    assert np.array_equal(ids, oi)
    assert dists.tobytes() == od.tobytes()
    # (in 64 bits, no query of the other laws comes within the error bound of its last candidate)
    assert fused == 1 and redone == (Q if law in ("row_scales", "huge_row") else 0)


@pytest.mark.parametrize("n,dim,Q,k,metric,scale_q,scale_b,redone", [
    (9000, 24, 40, 10, "l2", 1e18, 1.0, "all"),     # finite norms beyond a power of two of 2^-40 for the halves
    (20483, 24, 1030, 10, "ip", 1e18, 1.0, "all"),  # (two passes over the base)
    (9000, 24, 40, 10, "ip", 1e20, 1.0, "all"),     # |q|^2 overflows, every product is finite
    (9000, 24, 40, 10, "ip", 1.0, 1e20, "all"),     # |b|^2 overflows for every point
    (9000, 24, 40, 10, "l2", 1e17, 1e17, "few"),    # the screening vouches: its products are right at this scale
    (9000, 24, 40, 10, "ip", 1e18, 1e18, "few"),
    (9000, 24, 40, 10, "l2", 7e17, 7e17, "few"),
])
def test_screening_answers_for_large_magnitudes(orc, n, dim, Q, k, metric, scale_q, scale_b, redone):
    """Every component is finite and so is every distance: k neighbours, the oracle's, whatever the screening can
    vouch for.  Fused screening, screening through the matrix and the exact passes alike."""
    m = capi.IP if metric == "ip" else capi.L2
    base = synth.gaussian_matrix(n, n, dim) * np.float32(scale_b)
    q = synth.shifted_queries(Q, dim, 13, 14, 15) * np.float32(scale_q)
    oi, od = orc.bruteforce(base, q, k, m, order=SEQ)
    assert np.isfinite(od).all() and (oi >= 0).all()
    idx = capi.Index(base, None, None, m)
    for mode in (0, 2, 1):
        idx.bruteforce_exact_only(mode)
        ids, dists, _ = idx.bruteforce(q, k)
        assert np.array_equal(ids, oi) and dists.tobytes() == od.tobytes(), "mode %d" % mode
        if mode != 1:
            count = idx.bruteforce_last_redone()
            assert count == Q if redone == "all" else count <= Q // 4
    idx.close()


@pytest.mark.parametrize("metric", ["l2", "ip"])
def test_screening_of_distances_below_the_normal_range(orc, metric):
    """Products and squares of a few units of 2^-149: the reference order rounds each of them, the screening rounds
    their sum, and the two differ by more than neighbouring ranks do."""
    n, dim, Q, k = 9000, 24, 40, 200
    base = synth.gaussian_matrix(n, n, dim) * np.float32(5e-23)
    q = synth.shifted_queries(Q, dim, 13, 14, 15) * np.float32(5e-23)
    m = capi.IP if metric == "ip" else capi.L2
    oi, od = orc.bruteforce(base, q, k, m, order=SEQ)
    assert 0.0 < np.abs(od).max() < 1.2e-38
    idx = capi.Index(base, None, None, m)
    for mode in (0, 2, 1):
        idx.bruteforce_exact_only(mode)
        ids, dists, _ = idx.bruteforce(q, k)
        assert np.array_equal(ids, oi) and dists.tobytes() == od.tobytes(), "mode %d" % mode
    idx.close()


def test_randomised_knn_problems_equal_the_oracle(orc):
    """Seeded random sizes, k, metrics, tombstones and laws of the data (ties on a lattice, repeated vectors, large
    and small magnitudes, a common offset that makes the screening's error bound bite): the screened path and the
    exact-only path both return the oracle's ids and distance bits; so does the screening with its candidates
    selected from the distance matrix instead of inside the kernel."""
    redone = fused = unfused = 0
    for c in range(80):
        rng = np.random.RandomState(7000 + c)
        n = int(rng.choice([50, 129, 300, 1000, 4097, 10000, 30000]))
        dim = int(rng.choice([4, 8, 12, 20, 32, 64, 100, 128, 200, 256, 512]))
        Q = int(rng.choice([1, 5, 37, 128, 129, 300]))
        k = int(rng.choice([1, 2, 10, 32, 64, 100, 129, 300]))
        metric = capi.IP if rng.rand() < 0.35 else capi.L2
        tomb = rng.rand() < 0.3
        kind = str(rng.choice(["gauss", "lattice", "dups", "big", "tiny", "offset"]))
        while n * dim * Q > 1e9:
            Q = max(1, Q // 2)
        print("case", dict(c=c, n=n, dim=dim, Q=Q, k=k, metric=metric, tomb=tomb, kind=kind), flush=True)
        base = synth.gaussian_matrix(2000 + c, n, dim)
        q = synth.shifted_queries(Q, dim, 3 + c, 4 + c, 5 + c)
        if kind == "lattice":
            base, q = np.round(base), np.round(q)
        elif kind == "dups":
            base[n // 2:] = base[:n - n // 2]
        elif kind == "big":
            base, q = base * 1000.0, q * 1000.0
        elif kind == "tiny":
            base, q = base * 1e-3, q * 1e-3
        elif kind == "offset":
            base, q = base + 50.0, q + 50.0
        base, q = base.astype(np.float32), q.astype(np.float32)
        if metric == capi.IP and kind in ("gauss", "dups"):
            base, q = synth.normalize_rows(base), synth.normalize_rows(q)
        mask = synth.tombstone_mask(n, 77 + c, int(rng.choice([2, 3, 10]))) if tomb else None
        oi, od = orc.bruteforce(base, q, k, metric, deleted=mask, order=SEQ)
        idx = capi.Index(base, None, None, metric)
        if tomb:
            idx.set_deleted(mask)
        for mode in (0, 2, 1):
            idx.bruteforce_exact_only(mode)
            ids, dists, _ = idx.bruteforce(q, k, have_delete=tomb)
            redone += idx.bruteforce_last_redone() if mode == 0 else 0
            if mode == 0 and n >= 8192 and k + 32 <= 1024:
                fused += idx.bruteforce_last_fused()
                unfused += 1 - idx.bruteforce_last_fused()
            else:
                assert idx.bruteforce_last_fused() == 0
            assert np.array_equal(ids, oi) and dists.tobytes() == od.tobytes(), "mode %d" % mode
        idx.close()
    print("selection inside the kernel: %d cases, handed to the distance matrix: %d" % (fused, unfused), flush=True)
    assert redone > 0  # some of these queries went through the exact passes after the screening
    assert fused > 0


def test_bruteforce_ties_are_ordered_by_id(orc):
    # integer lattice: many exactly equal distances, including across the k-th place
    side = 7
    grid = np.stack(np.meshgrid(*[np.arange(side)] * 4, indexing="ij"), -1).reshape(-1, 4).astype(np.float32)
    q = np.array([[3, 3, 3, 3], [0, 0, 0, 0], [2.5, 3, 1, 6]], np.float32)
    idx = capi.Index(grid, ring(grid.shape[0]), np.array([0], np.int32))
    redone = 0
    for k in (1, 9, 33, 81, 200):
        ids, dists, _ = idx.bruteforce(q, k)
        redone += idx.bruteforce_last_redone()
        oi, od = orc.bruteforce(grid, q, k, order=SEQ)
        assert np.array_equal(ids, oi) and dists.tobytes() == od.tobytes()
        d2 = ((grid[ids] - q[:, None, :]) ** 2).sum(-1)
        assert np.array_equal(d2, dists)
        # within equal distances ids ascend
        for r in range(q.shape[0]):
            same = np.diff(dists[r]) == 0
            assert (np.diff(ids[r])[same] > 0).all()
    assert redone > 0  # ties across the last candidate's place: the screening hands those queries over
    idx.close()


def test_bruteforce_rows_with_thousands_of_ties_and_large_k(orc):
    # 30 000 points on a 3 x 3 x 3 x 3 lattice: every distance value is shared by hundreds of points, so the
    # candidates at the selection threshold outgrow the fast path's buffer and the radix path takes the rows;
    # k above 1024 goes to the radix path directly
    rng = np.random.RandomState(3)
    pts = rng.randint(0, 3, (30000, 4)).astype(np.float32)
    q = np.array([[1, 1, 1, 1], [0, 0, 0, 0], [0.5, 2, 1, 0], [7, 7, 7, 7]], np.float32)
    idx = capi.Index(pts, None, None)
    for k in (1, 100, 1000, 1025, 2000):
        ids, dists, _ = idx.bruteforce(q, k)
        oi, od = orc.bruteforce(pts, q, k, order=SEQ)
        assert np.array_equal(ids, oi) and dists.tobytes() == od.tobytes()
    # a mix in one batch: rows with few ties next to rows with many
    mixed = np.concatenate([pts[:15000], synth.gaussian_matrix(5, 15000, 4)])
    idx2 = capi.Index(mixed, None, None)
    q2 = np.concatenate([q, synth.gaussian_matrix(6, 4, 4)])
    ids, dists, _ = idx2.bruteforce(q2, 64)
    oi, od = orc.bruteforce(mixed, q2, 64, order=SEQ)
    assert np.array_equal(ids, oi) and dists.tobytes() == od.tobytes()
    idx.close(), idx2.close()


def test_bruteforce_candidate_lists_that_overflow_go_through_the_matrix(orc):
    """The selection inside the matrix-core kernel keeps what does not exceed a bound taken from a sample of the base.
    Where that is more than a list holds -- most of the base at one and the same distance, or a sample that is
    tombstoned away so that no bound exists -- the call falls back to the distance matrix, with the same result."""
    n, dim, k = 20000, 16, 10
    rng = np.random.RandomState(5)
    q = synth.gaussian_matrix(8, 7, dim)
    # (a) all but 50 rows are the same vector: every one of them ties at the bound
    base = np.ones((n, dim), np.float32)
    base[rng.choice(n, 50, replace=False)] = synth.gaussian_matrix(9, 50, dim)
    idx = capi.Index(base, None, None)
    ids, dists, _ = idx.bruteforce(q, k)
    assert idx.bruteforce_last_fused() == 0
    oi, od = orc.bruteforce(base, q, k, order=SEQ)
    assert np.array_equal(ids, oi) and dists.tobytes() == od.tobytes()
    idx.close()
    # (b) everything but the last 300 ids is tombstoned: the sample holds fewer live points than candidates are kept
    base = synth.gaussian_matrix(10, n, dim)
    mask = np.zeros((n + 31) // 32, np.uint32)
    dead = np.arange(n - 300)
    np.bitwise_or.at(mask, dead >> 5, (np.uint32(1) << (dead & 31).astype(np.uint32)))
    idx = capi.Index(base, None, None)
    idx.set_deleted(mask)
    ids, dists, _ = idx.bruteforce(q, k, have_delete=True)
    assert idx.bruteforce_last_fused() == 0
    oi, od = orc.bruteforce(base, q, k, deleted=mask, order=SEQ)
    assert np.array_equal(ids, oi) and dists.tobytes() == od.tobytes()
    assert (ids >= n - 300).all()
    idx.close()


def clustered(n, dim, size, Q, seed):
    """Clusters of `size` consecutive rows, well apart, and queries that belong to one each."""
    centres = 3.0 * synth.gaussian_matrix(seed, (n + size - 1) // size, dim)
    base = np.repeat(centres, size, axis=0)[:n] + synth.gaussian_matrix(seed + 1, n, dim)
    own = np.random.RandomState(seed).randint(0, centres.shape[0], Q)
    q = centres[own] + synth.gaussian_matrix(seed + 2, Q, dim)
    return base.astype(np.float32), q.astype(np.float32)


@pytest.mark.parametrize("n,size,Q", [
    (300000, 200, 1024),  # two passes whose first takes every 4th tile, after a sample of every 18th
    (20000, 64, 1024),    # every 4th and every 19th; clusters of half a tile
])
def test_two_screening_passes_over_a_base_stored_cluster_by_cluster(orc, n, size, Q):
    """The tiles of the first pass are not those of the sample: it may meet nothing of the cluster that a query's bound
    came from.  The bound still holds, and no list overflows."""
    dim, k = 16, 10
    base, q = clustered(n, dim, size, Q, 900)
    idx = capi.Index(base, None, None)
    ids, dists, _ = idx.bruteforce(q, k)
    fused = idx.bruteforce_last_fused()
    idx.close()
    oi, od = orc.bruteforce(base, q, k, order=SEQ)
    assert np.array_equal(ids, oi) and dists.tobytes() == od.tobytes()
    assert fused == 1


def test_bruteforce_segments(orc):
    # more base points than one pass holds (4M): per-segment winners are merged
    n, dim, Q, k = 5 * 1000 * 1000, 8, 40, 50
    base = workloads.gaussian_base(61, n, dim)
    q = synth.shifted_queries(Q, dim, 6, 7, 8)
    idx = capi.Index(base, ring(n), np.array([0], np.int32))
    ids, dists, _ = idx.bruteforce(q, k)
    idx.close()
    oi, od = orc.bruteforce(base, q, k, order=SEQ)
    assert np.array_equal(ids, oi) and dists.tobytes() == od.tobytes()


def test_bruteforce_ground_truth_at_full_size(orc):
    import torch
    n, dim, Q, k = 1000000, 200, 10000, 100
    base = workloads.gaussian_base(2001, n, dim)
    q = synth.shifted_queries(Q, dim, 2002, 2003, 2004)
    idx = capi.Index(base, ring(n), np.array([0], np.int32))
    ids, dists, t = idx.bruteforce(q, k)
    assert idx.bruteforce_last_fused() == 1 and idx.bruteforce_last_redone() == 0
    idx.bruteforce_exact_only(2)
    ids_m, dists_m, t_m = idx.bruteforce(q, k)
    idx.bruteforce_exact_only(0)
    assert np.array_equal(ids_m, ids) and dists_m.tobytes() == dists.tobytes()
    print("candidates selected inside the kernel: %.3f s; from the distance matrix: %.3f s" % (t, t_m), flush=True)
    pairs = float(Q) * n * dim
    print("brute force 10k x 1M x 200: %.3f s, %.2f T pair-dims/s (%.1f TFLOP/s at 3 flop per pair-dim)" %
          (t, pairs / t / 1e12, 3 * pairs / t / 1e12), flush=True)
    assert (np.diff(dists, axis=1) >= 0).all()
    sub = np.arange(0, Q, 313)
    t0 = time.perf_counter()
    oi, od = orc.bruteforce(base, q[sub], k, order=SEQ)
    t_cpu = time.perf_counter() - t0
    print("oracle on %d host threads: %d queries in %.2f s = %.0f queries/s (device: %.0f queries/s)" %
          (orc.max_threads(), len(sub), t_cpu, len(sub) / t_cpu, Q / t), flush=True)
    assert np.array_equal(ids[sub], oi) and dists[sub].tobytes() == od.tobytes()
    # agrees with a matmul-based top-k (|b|^2 - 2 q.b, another arithmetic altogether) up to near-ties
    tb, tq = torch.from_numpy(base).cuda(), torch.from_numpy(q[sub]).cuda()
    gt = torch.topk((tb * tb).sum(1)[None, :] - 2.0 * (tq @ tb.T), k, dim=1, largest=False).indices.cpu().numpy()
    del tb, tq
    agree = np.mean([len(set(a.tolist()) & set(b.tolist())) for a, b in zip(ids[sub], gt)]) / k
    assert agree > 0.999
    # device-pointer entry, and the gt-file layout on disk
    tq = torch.from_numpy(q[:256]).cuda()
    d_ids = torch.empty((256, k), dtype=torch.int32, device="cuda")
    idx.bruteforce_device(tq.data_ptr(), d_ids.data_ptr(), None, 256, k)
    assert np.array_equal(d_ids.cpu().numpy(), ids[:256])
    idx.close()


@pytest.mark.parametrize("law,metric,dim,k,dele", [
    ("gauss", "l2", 100, 100, False), ("gauss", "l2", 120, 1, True), ("cone", "ip", 132, 10, False),
    ("cone", "ip", 144, 200, True),
    ("offset", "l2", 100, 100, False),   # norms far beyond the spread: one product cannot tell the rows apart
    ("pairs", "l2", 100, 40, False),     # every row twice, and queries among them: ties at every place
    ("lattice", "l2", 100, 10, False),   # exact in halves, thousands of equal distances
    ("scales", "l2", 100, 20, False),    # rows of norms 1e-3 .. 1e3: a few decide the bound for all
    ("tiny", "ip", 100, 20, False),      # components below what scaled halves hold
    ("crowd", "l2", 100, 10, False),     # a few queries among rows that one product, or three, cannot tell apart
])
def test_screening_on_one_product_answers_what_the_plain_passes_answer(law, metric, dim, k, dele):
    """Batches large enough to be screened on one product of halves per pair (1e11 pair dimensions; their last stage of
    32 dimensions is whole, half or less): ids and distance bits are those of the search that measures every pair in
    the reference's order, whether the candidates vouch for them or the queries go on to three products and beyond."""
    n, Q = 300000, 3400
    assert Q * n * dim >= 1e11
    rng = np.random.RandomState(dim + k)
    base = synth.gaussian_matrix(5, n, dim)
    q = synth.shifted_queries(Q, dim, 6, 7, 8)
    if law == "cone":
        base = synth.normalize_rows(base)
        q = synth.normalize_rows(q + 3.0)
    if law == "offset":
        base += np.float32(30.0)
        q += np.float32(30.0)
    if law == "pairs":
        base[1::2] = base[::2]
        q[::2] = base[rng.choice(n, Q // 2, replace=False)]
    if law == "lattice":
        base = rng.randint(-2, 3, (n, dim)).astype(np.float32)
        q = rng.randint(-2, 3, (Q, dim)).astype(np.float32)
    if law == "scales":
        base *= (10.0 ** rng.randint(-3, 4, (n, 1))).astype(np.float32)
    if law == "tiny":
        base[:, 1:] *= np.float32(1e-7)
    if law == "crowd":
        for at, width in ((1000, 5e-3), (2000, 1e-4)):
            base[at:at + 500] = base[at] + np.float32(width) * base[at:at + 500]
            q[at:at + 40] = base[at] + np.float32(0.5) * q[at:at + 40]
    idx = capi.Index(base, None, None, metric=capi.IP if metric == "ip" else capi.L2)
    if dele:
        idx.mark_deleted(rng.choice(n, n // 5, replace=False).astype(np.int32))
    print("one product", law, metric, dim, k, dele, flush=True)
    ids, dists, _ = idx.bruteforce(q, k, have_delete=dele)
    redone, handed_on = idx.bruteforce_last_redone(), idx.bruteforce_last_handed_on()
    # which way it went: on one product, on to three by the sample's word, or on to three query by query
    if law in ("offset", "scales", "tiny"):
        assert handed_on == -1
    elif law == "crowd":
        assert 40 <= redone < handed_on <= 80
    else:
        assert handed_on >= 0
    idx.bruteforce_exact_only(2)
    ids3, dists3, _ = idx.bruteforce(q, k, have_delete=dele)
    assert idx.bruteforce_last_redone() == redone  # what one product leaves open three decide as they did
    idx.bruteforce_exact_only(True)
    want_ids, want_d, _ = idx.bruteforce(q, k, have_delete=dele)
    idx.close()
    assert np.array_equal(ids, want_ids) and dists.tobytes() == want_d.tobytes()
    assert np.array_equal(ids3, want_ids) and dists3.tobytes() == want_d.tobytes()


@pytest.mark.parametrize("Q", [1, 3, 255, 257, 1024, 1025, 4500])
@pytest.mark.parametrize("metric,dim,k", [("l2", 4, 1), ("ip", 12, 10), ("l2", 100, 10), ("ip", 260, 33), ("l2", 516, 5)])
def test_prepared_queries_at_the_edges_of_tiles_and_flags(Q, metric, dim, k):
    """Batches about the query tile of 256, the 1024 queries whose flags go to pinned memory and the 2048 and 4096 of a block
    of the screening; dimensions short of a stage of 16 and beyond the 64 lanes that read a row.  Twice on one index (the
    counters start at zero again), and with every second base row equal, where lists overflow or leave ties open: ids and
    distance bits are those of the search that measures every pair."""
    rng = np.random.RandomState(Q + dim)
    base = synth.gaussian_matrix(9, 12000, dim)
    q = synth.shifted_queries(Q, dim, 6, 7, 8)
    for twins in (False, True):
        if twins:
            base[1::2] = base[:1]
            q[::3] = base[rng.choice(12000, len(q[::3]))]
        idx = capi.Index(base, None, None, metric=capi.IP if metric == "ip" else capi.L2)
        print("prepared", Q, metric, dim, k, twins, flush=True)
        first = idx.bruteforce(q, k)
        again = idx.bruteforce(q, k)
        fused = idx.bruteforce_last_fused()
        idx.bruteforce_exact_only(True)
        want_ids, want_d, _ = idx.bruteforce(q, k)
        idx.close()
        assert fused or twins
        for ids, dists, _ in (first, again):
            assert np.array_equal(ids, want_ids) and dists.tobytes() == want_d.tobytes()
