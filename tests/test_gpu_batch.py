"""GPU tests of the launch variants that must not change any result: the
hipGraph-replayed loop, the tile-queue launch shapes, and the batched solve
(many instances, several streams, optional graph) against single solves."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)


@pytest.fixture(scope="module")
def S():
    assert torch.cuda.is_available()
    from egg_sync import solver
    return solver


def _same(a, b):
    assert a["stats"]["iterations"] == b["stats"]["iterations"]
    assert np.array_equal(a["labels"], b["labels"])
    assert np.array_equal(a["X"].view(np.uint32), b["X"].view(np.uint32))


def test_graph_replays_match_eager(S):
    from egg_sync import data
    X, eps = data.config1(seed=11, n=60000)
    ref = S.solve(X, eps, iters_per_sync=2)
    _say("eager:", ref["stats"]["iterations"], "iterations")
    for rep in range(3):
        g = S.solve(X, eps, iters_per_sync=2, use_graph=True)
        _same(ref, g)
        e = S.solve(X, eps, iters_per_sync=3)      # eager work between replays
        _same(ref, e)
    X2, _ = data.config1(seed=12, n=60000)         # same shape, new data: graph reused
    _same(S.solve(X2, eps, iters_per_sync=2), S.solve(X2, eps, iters_per_sync=2, use_graph=True))


def test_graph_timing_and_sync_mode(S):
    from egg_sync import data, _native as nat
    X, eps = data.config0(seed=0)
    a = S.solve(X, eps, stop_rule=nat.STOP_RC)
    b = S.solve(X, eps, stop_rule=nat.STOP_RC, use_graph=True, timing=True, iters_per_sync=5)
    _same(a, b)
    assert b["stats"]["stage_ms"][2] > 0


@pytest.mark.parametrize("qt,qb", [(64, 0), (128, 0), (192, 0), (256, 7), (64, 1), (256, 300)])
def test_queue_launch_shapes_are_bitwise_neutral(S, qt, qb):
    from egg_sync import data
    X, eps = data.config1(seed=13, n=40000)
    ref = S.solve(X, eps)
    _same(ref, S.solve(X, eps, queue_threads=qt, queue_blocks=qb))


@pytest.mark.parametrize("gw", [2, 4, 8, 3])
def test_tile_groups_change_only_rounding(S, O, gw):
    """Which runs share a wavefront decides which sub-cells it streams point by
    point, so tile groups change the order of FP32 additions, nothing else:
    iterations, counts and partitions stay those of the oracle."""
    from egg_sync import data
    cases = [(*data.config1(seed=14, n=40000),),
             (data.gaussian_blobs(6000, 5, 4, seed=15, center_lo=0.2, center_hi=0.8,
                                  sigma=0.03, noise=0.05), 0.1),
             (data.config2(n=5000)[0], 0.1)]
    for X, eps in cases:
        a, b = S.solve(X, eps, tile_group=1), S.solve(X, eps, tile_group=gw)
        assert a["stats"]["iterations"] == b["stats"]["iterations"]
        assert O.same_partition(a["labels"], b["labels"])
        assert np.abs(a["X"] - b["X"]).max() <= 1e-5
        it_a = S.iteration(X, eps)
        o = O.egg_iteration(X, eps)
        for k in ("N", "half", "border", "synced"):
            assert np.array_equal(it_a[k], o[k]), k


def _mixed_instances():
    from egg_sync import data
    rng = np.random.default_rng(5)
    sets = []
    for i, (n, d) in enumerate([(3000, 2), (20000, 3), (500, 5), (8000, 8), (1, 3), (12000, 3)]):
        sets.append(data.gaussian_blobs(n, d, int(rng.integers(2, 8)), seed=100 + i,
                                        center_lo=0.2, center_hi=0.8, sigma_lo=0.01,
                                        sigma_hi=0.04, sizes="equal", noise=0.03))
    eps = [[0.05, 0.02], [0.02], [0.1], [0.1, 0.2], [0.05], [0.01, 0.05]]
    return sets, eps


@pytest.mark.parametrize("streams,graph", [(1, False), (3, False), (4, True), (2, True),
                                           (24, False), (24, True)])
def test_batch_equals_single_solves(S, streams, graph):
    sets, eps = _mixed_instances()
    D, specs = S.pack_instances(sets, eps)
    specs.insert(3, (0, 0, 2, 0.05))               # an empty instance in the middle
    r = S.solve_batch(D, specs, streams=streams, use_graph=graph, iters_per_sync=3)
    _say(f"batch streams={streams} graph={graph}: {len(specs)} instances, "
         f"{r['stats']['total_ms']:.1f} ms, max iterations {r['stats']['iterations']}")
    k = 0
    for X, es in zip(sets, eps):
        for e in es:
            if k == 3:
                assert r["labels"][k].size == 0 and r["results"][k]["iterations"] == 0
                k += 1
            single = S.solve(X, e)
            assert r["results"][k]["iterations"] == single["stats"]["iterations"], k
            assert r["results"][k]["n_clusters"] == single["stats"]["n_clusters"], k
            assert np.array_equal(r["labels"][k], single["labels"]), k
            assert np.array_equal(r["X"][k].view(np.uint32), single["X"].view(np.uint32)), k
            k += 1
    assert k == len(specs)


def test_batch_sync_mode_equals_single(S):
    from egg_sync import data, _native as nat
    sets = [data.config0(seed=s, n=n)[0] for s, n in ((0, 2000), (1, 700), (2, 1500))]
    D, specs = S.pack_instances([(x, 0.05) for x in sets])
    r = S.solve_batch(D, specs, stop_rule=nat.STOP_RC, streams=2)
    for k, X in enumerate(sets):
        single = S.solve(X, 0.05, stop_rule=nat.STOP_RC)
        assert r["results"][k]["iterations"] == single["stats"]["iterations"]
        assert np.array_equal(r["labels"][k], single["labels"])


def test_batch_rejects_out_of_range_input(S):
    from egg_sync import _native as nat
    D = torch.rand(3000, device="cuda")
    D[2500] = 1.5
    with pytest.raises(nat.EggSyncError):
        S.solve_batch(D, [(0, 1000, 2, 0.05), (2000, 500, 2, 0.05)])
    r = S.solve_batch(D, [(0, 1000, 2, 0.05)])     # the bad value lies outside this instance
    assert r["labels"][0].shape == (1000,)


def _passes_match_oracle_along_gpu_trajectory(S, O, X, e, iters):
    """Each GPU pass equals the oracle's pass from the same (GPU) state."""
    prev = X
    for t in range(1, iters + 1):
        cur = S.solve(X, e, max_iter=t)["X"]
        ref = O.egg_iteration(prev, e)["X_next"]
        assert np.abs(cur - ref).max() <= 1e-6, t
        prev = cur


def test_batch_graph_with_wide_keys(S):
    """64 instances x 16 iterations whose radix sorts take 22 passes (175 key
    bits): counted as 81 kernels an iteration, 82,944 in all, past the largest
    batched graph, so it launches plainly and gives what one instance gives."""
    rng = np.random.default_rng(5)
    n, d, eps = 24577, 20, 0.1
    X = rng.random((n // 2 + 1, d))
    X = np.repeat(X, 2, axis=0)[:n] + 0.002 * rng.random((n, d))
    X = np.clip(X, 0, 1).astype(np.float32)
    one = S.solve(X, eps, max_iter=3)
    D, specs = S.pack_instances([X], [[eps] * 64])
    r = S.solve_batch(D, specs, streams=4, use_graph=True, iters_per_sync=16, max_iter=3)
    for k in range(64):
        assert r["results"][k]["iterations"] == one["stats"]["iterations"], k
        assert np.array_equal(r["labels"][k], one["labels"]), k
        assert np.array_equal(r["X"][k].view(np.uint32), one["X"].view(np.uint32)), k


def test_batch_config3_sample_against_oracle(S, O):
    """Iterations and partitions equal the oracle's.  Final positions agree to
    1e-5 unless the trajectory is sensitive to last-bit differences: a pair at
    distance eps +- 1 ulp is inside the eps-ball for one state and outside for
    the other, and the two runs then follow different (equally valid) paths to
    the same partition.  For those instances every GPU pass is checked against
    the oracle's pass from the same state instead."""
    from egg_sync import data
    from egg_sync.metrics import same_partition
    inst = data.config3_instances(seed=3, count=6, n_lo=1000, n_hi=6000)
    D, specs = S.pack_instances(inst, [list(data.CONFIG3_EPS)] * len(inst))
    r = S.solve_batch(D, specs, streams=4, use_graph=True)
    k = 0
    for X in inst:
        for e in data.CONFIG3_EPS:
            o = O.egg_solve(X, e)
            assert r["results"][k]["iterations"] == o["iterations"], (k, X.shape, e)
            assert same_partition(r["labels"][k], o["labels"]), (k, X.shape, e)
            err = float(np.abs(r["X"][k] - o["X"]).max())
            if err > 1e-5:
                _say(f"instance {k} {X.shape} eps={e}: final positions differ by {err:.3g}; "
                     "checking every pass along the GPU trajectory")
                _passes_match_oracle_along_gpu_trajectory(S, O, X, e, o["iterations"])
            k += 1


def test_autotuner_checks_results_and_caches(S, tmp_path, monkeypatch):
    from egg_sync import autotune
    monkeypatch.setenv("EGG_SYNC_TUNE_CACHE", str(tmp_path / "tune.json"))
    sets, eps = _mixed_instances()
    D, specs = S.pack_instances(sets, eps)
    space = {"streams": [2, 4], "use_graph": [False, True], "iters_per_sync": [4, 2]}
    best, t, table = autotune.tune_batch(D, specs, repeats=1, space=space, log=_say)
    assert len(table) >= 3 and t > 0
    assert autotune.cached(autotune.batch_signature(specs)) == best
    r = S.solve_batch(D, specs, **best)
    assert r["results"][0]["iterations"] > 0


def test_experiment_harness_records():
    from egg_sync import experiments as E
    recs = E.run("n", [2000, 4000], rounds=2, d=2, eps=0.05)
    assert len(recs) == 4
    for r in recs:
        assert r["running_time"] > 0 and r["iterations"] >= 1 and r["space"] > 0
        assert list(r["stage_times"]) == E.STAGES
        assert len(r["itr_times"]) == r["iterations"]
    recs = E.run("d", [3, 8, 20], rounds=1, n=3000, eps=0.2)
    assert [r["d"] for r in recs] == [3, 8, 20]


def test_batch_config3_slowest_instance_against_oracle(S, O):
    """The slowest instance of the 64-instance batched workload (n=165,583, d=2,
    eps=0.1; the oracle needs 11,608 iterations), against the committed oracle
    run (tests/golden/make_oracle_fixtures.py c3_tail).  Over ~11,600 passes the
    last-bit differences of the summation order make the trajectory take a
    different, equally valid path (see the test above), so the stop may come
    one pass earlier or later; the partition must be the same, and at
    checkpoints along the GPU trajectory and at its end a GPU pass equals the
    oracle's pass from the same state bit for bit in every integer output."""
    from conftest import golden
    from egg_sync import data
    from egg_sync.metrics import same_partition
    g = golden("c3_tail_oracle")
    X = data.config3_instances(seed=3, count=64)[27]
    eps = 0.1
    assert X.shape == (165583, 2)
    D, specs = S.pack_instances([X], [[eps]])
    _say("config3 slowest instance, batched solve")
    r = S.solve_batch(D, specs)
    it = r["results"][0]["iterations"]
    _say("iterations", it, "oracle", int(g["iterations"]))
    assert r["results"][0]["status"] == 0
    assert abs(it - int(g["iterations"])) <= 1
    assert same_partition(r["labels"][0], g["labels"])
    a = S.solve(X, eps)
    assert a["stats"]["iterations"] == it and np.array_equal(a["labels"], r["labels"][0])
    for t in (1000, 6000, it - 1):
        Xt = S.solve(X, eps, max_iter=t)["X"]
        _say("pass from the GPU state after", t, "iterations")
        ga = S.iteration(Xt, eps)
        gb = O.egg_iteration(Xt, eps)
        for k in ("order", "N", "half", "border", "synced"):
            assert np.array_equal(ga[k], gb[k]), (t, k)
        assert (ga["flag_local"], ga["flag_final"]) == (gb["flag_local"], gb["flag_final"]), t
        # Positions: within 1e-6 of the FP64 oracle's pass from the same state.
        # Where the FP32 oracle's plain left-to-right sum over up to ~40,000
        # neighbours drifts further (7e-6 measured at t=1000), the GPU (sums
        # split per sub-cell, runs weighted by length) stays within 1e-7 of
        # FP64, so it may differ from the FP32 oracle by that oracle's own error.
        x64 = O.egg_solve(Xt, eps, max_iter=1, fp64=True)["X"].astype(np.float64)
        err64 = np.abs(ga["X_next"] - x64)
        _say(f"  max |gpu - fp64| {err64.max():.3g}, "
             f"max |fp32 oracle - fp64| {np.abs(gb['X_next'] - x64).max():.3g}")
        assert err64.max() <= 1e-6, t
        assert (np.abs(ga["X_next"] - gb["X_next"]) <= 1e-6 + np.abs(gb["X_next"] - x64)).all(), t
    # the state the GPU stopped on is one the oracle's stop rule also accepts
    assert gb["flag_final"] == 1
    assert np.abs(ga["X_next"] - a["X"]).max() <= 1e-6


def test_launch_shapes_bitwise_neutral_at_full_size(S):
    """n = 1,000,000 (config 1): dense clusters make streamed ranges of >= 4096
    runs, which are split into units summed in fixed point by whichever
    wavefront takes them; the result must not depend on the launch shape."""
    from egg_sync import data
    X, eps = data.config1()
    ref = S.solve(X, eps)
    for qt, qb in ((64, 0), (128, 512)):
        _say("config1 queue shape", qt, qb)
        _same(ref, S.solve(X, eps, queue_threads=qt, queue_blocks=qb))


def test_config3_slowest_instance_where_trajectories_part(S, O):
    """Why the slowest config-3 instance may stop a pass earlier or later than
    the oracle: from the GPU's state after 8,607 passes the GPU and the oracle
    step side by side, each from its own previous state.  Every pass takes the
    same per-point decisions (N, half, border, synced, both flags) until a
    cluster of ~20,000 equal points drifting across a cell face enters the
    reference's +-1e-5 border band (EGG_SynC.cu:590-595) at different passes:
    the two trajectories' positions part by the FP32 oracle's rounding (it adds
    the cluster's equal terms one by one; the GPU weights the run by its
    length), 3.3e-5 after ~2,600 passes.  No eps or eps/2 test decides
    differently first: N is equal at the first differing pass, and every point
    whose border flag differs has the band's edge between its two positions."""
    from egg_sync import data
    f32 = np.float32
    X = data.config3_instances(seed=3, count=64)[27]
    eps = 0.1
    K = 8607
    cs = float(f32(np.sqrt((float(f32(eps)) / 2) ** 2 / 2)))
    X0 = S.solve(X, eps, max_iter=K)["X"]
    _say("slowest instance: GPU and oracle from the GPU state after", K, "passes")

    def per_point(r, f):
        a = np.empty_like(r[f])
        a[r["order"]] = r[f]
        return a

    def band_margin(x):
        # distance of the nearest coordinate to the edge of a face's +-1e-5 band
        xd = x.astype(np.float64)
        face = np.round(xd / cs) * cs
        return (np.abs(np.abs(xd - face) - 1e-5)).min(axis=1)

    Xg, og, Xo, oo = X0, None, X0, None
    for k in range(4000):
        rg = S.iteration(Xg, eps, og)
        ro = O.egg_iteration(Xo, eps, oo)
        diff = [f for f in ("N", "half", "border", "synced")
                if not np.array_equal(per_point(rg, f), per_point(ro, f))]
        flags_equal = (rg["flag_local"], rg["flag_final"]) == (ro["flag_local"], ro["flag_final"])
        if diff or not flags_equal:
            gap = float(np.abs(Xg - Xo).max())
            _say(f"  first differing pass {K + k + 1}: {diff}, positions {gap:.3g} apart")
            assert "N" not in diff and flags_equal
            assert "border" in diff and gap <= 1e-4
            pts = np.nonzero(per_point(rg, "border") != per_point(ro, "border"))[0]
            _say(f"  {len(pts)} points change border status")
            m = np.minimum(band_margin(Xg[pts]), band_margin(Xo[pts]))
            # (1e-6: the faces' own FP32 placement, id * cs)
            assert np.all(m <= np.abs(Xg[pts] - Xo[pts]).max(axis=1) + 1e-6)
            return
        if rg["flag_final"]:
            _say(f"  both stop at pass {K + k + 1} with equal decisions throughout")
            return
        Xg, og, Xo, oo = rg["X_next"], rg["order"], ro["X_next"], ro["order"]
    pytest.fail("neither trajectory stopped")
