"""Batched cycle (all pairs x hypotheses in one launch per iteration, replayed
from a hipGraph) against the single-pair path and the oracle."""
import numpy as np
import pytest

import oracle
from conftest import print_case
from lowcost3dreconstruction_amd import synth

pytestmark = pytest.mark.gpu

KW = dict(max_corr_dist=0.01, max_iterations=60, transformation_epsilon=1e-9,
          euclidean_fitness_epsilon=1e-3)


@pytest.fixture(scope="module")
def small_cycle():
    cyc = synth.turntable_cycle(11, n_captures=6, yaw_step_deg=10.0, scale=1.5,
                                centre=(0.0, 0.0, -0.8))
    normals = [oracle.normals(c, 30)[0] for c in cyc.clouds]
    return cyc, normals


def single_pair(lcr, src, tgt, tn, guess):
    icp = lcr.IterativeClosestPoint(point_to_plane=True)
    icp.setInputSource(src)
    icp.setInputTarget(tgt, tn)
    icp.setMaxCorrespondenceDistance(KW["max_corr_dist"])
    icp.setMaximumIterations(KW["max_iterations"])
    icp.setTransformationEpsilon(KW["transformation_epsilon"])
    icp.setEuclideanFitnessEpsilon(KW["euclidean_fitness_epsilon"])
    icp.align(guess)
    return icp


def test_cycle_equals_single_pairs_bitwise(lcr, small_cycle):
    cyc, normals = small_cycle
    print_case(test="cycle_vs_single", pairs=len(cyc.pairs))
    c = lcr.Cycle(cyc.clouds, cyc.pairs, normals=normals, guesses=cyc.meta["prior"],
                  point_to_plane=True, **KW)
    c.run()
    r = c.results()
    for i, (s, t) in enumerate(cyc.pairs):
        icp = single_pair(lcr, cyc.clouds[s], cyc.clouds[t], normals[t], cyc.meta["prior"][i])
        np.testing.assert_array_equal(r["T"][i], icp.getFinalTransformation())
        assert r["iterations"][i] == icp.nr_iterations()
        assert r["state"][i] == icp.getConvergenceState()
        assert r["fitness"][i] == icp.getFitnessScore()


def test_cycle_matches_oracle_and_is_deterministic(lcr, small_cycle):
    cyc, normals = small_cycle
    print_case(test="cycle_oracle")
    c = lcr.Cycle(cyc.clouds, cyc.pairs, normals=normals, guesses=cyc.meta["prior"],
                  point_to_plane=True, **KW)
    c.run()
    r1 = c.results()
    c.run()  # graph replay
    r2 = c.results()
    np.testing.assert_array_equal(r1["T"], r2["T"])
    refs = oracle.icp_batch(cyc.clouds, normals, cyc.pairs, guesses=cyc.meta["prior"],
                            point_to_plane=True, **KW)
    for i, ref in enumerate(refs):
        er, et = synth.transform_error(r1["T"][i], ref["T"])
        assert er < 1e-6 and et < 1e-7, (i, er, et)
        assert r1["iterations"][i] == ref["iterations"]
        assert r1["state"][i] == ref["state"]


def test_cycle_device_normals(lcr, small_cycle):
    """Normals estimated on the device inside the cycle: each pair lands within the
    benchmark's aligned bar (0.05 deg / 0.2 mm) of the oracle run on oracle normals,
    and much closer on most pairs."""
    cyc, normals = small_cycle
    print_case(test="cycle_dev_normals")
    c = lcr.Cycle(cyc.clouds, cyc.pairs, guesses=cyc.meta["prior"], point_to_plane=True,
                  normals_k=30, **KW)
    c.run()
    r = c.results()
    refs = oracle.icp_batch(cyc.clouds, normals, cyc.pairs, guesses=cyc.meta["prior"],
                            point_to_plane=True, **KW)
    errs = np.array([synth.transform_error(r["T"][i], ref["T"]) for i, ref in enumerate(refs)])
    assert np.all(errs[:, 0] < np.deg2rad(0.05)) and np.all(errs[:, 1] < 2e-4), errs
    assert np.median(errs[:, 0]) < 1e-5


def test_cycle_hypotheses_select_best_fitness(lcr, small_cycle):
    cyc, normals = small_cycle
    H = 3
    rng = np.random.default_rng(5)
    guesses = []
    for i in range(len(cyc.pairs)):
        P = cyc.meta["prior"][i]
        guesses += [P, synth.perturb(rng, 4.0, 0.01) @ P, np.eye(4)]
    guesses = np.stack(guesses)
    print_case(test="cycle_hyp", hyp=H)
    c = lcr.Cycle(cyc.clouds, cyc.pairs, normals=normals, guesses=guesses, n_hyp=H,
                  point_to_plane=True, **KW)
    c.run()
    inst = c.instances()
    r = c.results()
    for i, (s, t) in enumerate(cyc.pairs):
        fits = inst["fitness"][i * H:(i + 1) * H]
        assert r["best_hyp"][i] == int(np.argmin(fits))
        np.testing.assert_array_equal(r["T"][i], inst["T"][i * H + r["best_hyp"][i]])
        for h in range(H):
            icp = single_pair(lcr, cyc.clouds[s], cyc.clouds[t], normals[t], guesses[i * H + h])
            np.testing.assert_array_equal(inst["T"][i * H + h], icp.getFinalTransformation())


def test_cycle_point_to_point_and_empty_cloud(lcr):
    p = synth.pair_ellipsoids(4, n_src=3000, n_tgt=3000)
    empty = np.zeros((0, 3), np.float32)
    print_case(test="cycle_p2p_empty")
    c = lcr.Cycle([p.src, p.tgt, empty], [(0, 1), (2, 1), (0, 2)], point_to_plane=False,
                  max_corr_dist=0.05, max_iterations=50)
    c.run()
    r = c.results()
    ref = oracle.icp(p.src, p.tgt, max_corr_dist=0.05, max_iterations=50)
    er, et = synth.transform_error(r["T"][0], ref["T"])
    assert er < 1e-6 and et < 1e-7
    assert r["iterations"][0] == ref["iterations"]
    # empty source or target: nothing runs, not converged (Registration::initCompute)
    assert not r["converged"][1] and r["iterations"][1] == 0
    assert not r["converged"][2] and r["iterations"][2] == 0


def test_autotune_keeps_results_and_caches(lcr, small_cycle, tmp_path):
    """The tuner only changes the launch shape: transforms agree with the default
    setting to rounding (the FP64 reduction order follows the tile size and the
    source's cell order; the rotation angle, an arccos of the trace, resolves only
    about 1e-8 rad near zero), and a second tuner on the same workload reads its
    choice back from the cache."""
    cyc, normals = small_cycle
    print_case(test="autotune")
    base = lcr.Cycle(cyc.clouds, cyc.pairs, normals=normals, guesses=cyc.meta["prior"],
                     point_to_plane=True, **KW)
    base.run()
    r0 = base.results()
    cache = tmp_path / "tune.txt"
    c = lcr.Cycle(cyc.clouds, cyc.pairs, normals=normals, guesses=cyc.meta["prior"],
                  point_to_plane=True, **KW)
    t = c.autotune(str(cache))
    assert t["from_cache"] == 0 and t["candidates"] == 30
    assert t["tile"] in (64, 128, 256) and t["precision_mode"] in (0, 1, 2, 3)
    assert 0 < t["best_ms"] <= t["default_ms"] * 1.5
    c.run()
    r1 = c.results()
    for a, b in zip(r0["T"], r1["T"]):
        er, et = synth.transform_error(a, b)
        assert er < 1e-7 and et < 1e-9
    np.testing.assert_array_equal(r0["state"], r1["state"])
    c2 = lcr.Cycle(cyc.clouds, cyc.pairs, normals=normals, guesses=cyc.meta["prior"],
                   point_to_plane=True, **KW)
    t2 = c2.autotune(str(cache))
    assert t2["from_cache"] == 1
    assert (t2["tile"], t2["precision_mode"], t2["cell_factor"]) == \
        (t["tile"], t["precision_mode"], t["cell_factor"])


def test_hypothesis_gate_keeps_the_seed_and_the_best_initial_pose(lcr, small_cycle):
    """With hyp_gate, each pair's hypotheses are scored by their source points
    within r at the initial pose (on a fixed subsample of at least 32 tiles of 64
    source points).  The first hypothesis (the plain seed) is always refined; of
    the others, the best-scoring one is refined too when it scores above the seed;
    the lower final fitness wins.  Each refined pose is bitwise the single-pair ICP
    from it.  Against the oracle's full inlier counts: a clear winner among the
    others (1.5x the runner-up) must be the one refined, otherwise the refined one
    has at least 2/3 of their best count.  The seed here is a 20 deg perturbation of
    the prior and the prior is hypothesis 1, so the gate must find it."""
    from lowcost3dreconstruction_amd.synth import perturb, rigid
    cyc, normals = small_cycle
    H = 4
    rng = np.random.default_rng(3)
    guesses = []
    for (s, _), P in zip(cyc.pairs, cyc.meta["prior"]):
        c = P[:3, :3] @ cyc.clouds[s].astype(np.float64).mean(axis=0) + P[:3, 3]
        C = rigid(np.eye(3), c)
        for h, ang in enumerate((20.0, None, 15.0, 25.0)):
            if ang is None:
                guesses.append(P)
            else:
                R = perturb(rng, ang, 0.0)
                while synth.rotation_error(R[:3, :3], np.eye(3)) < np.deg2rad(0.8 * ang):
                    R = perturb(rng, ang, 0.0)
                guesses.append(C @ R @ np.linalg.inv(C) @ P)
    guesses = np.stack(guesses)
    print_case(test="gate", pairs=len(cyc.pairs), hyp=H)
    c = lcr.Cycle(cyc.clouds, cyc.pairs, normals=normals, guesses=guesses, n_hyp=H,
                  point_to_plane=True, hyp_gate=True, **KW)
    c.run()
    r = c.results()
    inst = c.instances()
    for i, (s, t) in enumerate(cyc.pairs):
        counts = [int((oracle.correspondences(cyc.clouds[s], cyc.clouds[t], guesses[i * H + h],
                                              KW["max_corr_dist"])[0] >= 0).sum())
                  for h in range(H)]
        refined = [h for h in range(H) if inst["iterations"][i * H + h] > 0]
        assert refined[0] == 0 and len(refined) <= 2, (i, refined)
        others = np.array(counts[1:])
        order = np.argsort(others)[::-1] + 1
        if len(refined) == 2:
            alt = refined[1]
            if counts[order[0]] > 1.5 * counts[order[1]]:
                assert alt == order[0], (i, counts, alt)
            else:
                assert counts[alt] >= (2 / 3) * counts[order[0]], (i, counts, alt)
        else:
            # no other hypothesis beat the seed: the seed has a clear lead or a near tie
            assert counts[0] >= (2 / 3) * counts[order[0]], (i, counts)
        fits = [inst["fitness"][i * H + h] for h in refined]
        kept = int(r["best_hyp"][i])
        assert kept == refined[int(np.argmin(fits))]
        for h in refined:
            icp = single_pair(lcr, cyc.clouds[s], cyc.clouds[t], normals[t], guesses[i * H + h])
            np.testing.assert_array_equal(inst["T"][i * H + h], icp.getFinalTransformation())
            assert inst["fitness"][i * H + h] == icp.getFitnessScore()
        np.testing.assert_array_equal(c.initial_poses()[i * H:(i + 1) * H], guesses[i * H:(i + 1) * H])


def test_batch_of_more_than_33m_cells_equals_single_pairs(lcr):
    """Thin diagonal clouds whose boxes take the capped cell count: five of them hold
    more cells than one scan adds up without its extra pass (8192 tiles of 4096); a
    pair's own build stays below.  Bitwise the same transforms."""
    rng = np.random.default_rng(21)
    clouds = []
    for i in range(5):
        t = rng.uniform(0, 1, size=(830_000, 1))
        clouds.append((t * np.array([[1.0, 0.9, 0.8]]) + rng.normal(scale=2e-3, size=(len(t), 3))
                       + 1e-4 * i).astype(np.float32))
    print_case(test="large_scan")
    kw = dict(max_corr_dist=0.002, max_iterations=2, point_to_plane=False)
    c = lcr.Cycle(clouds, [(1, 0), (4, 3)], **kw)
    c.run()
    T = c.results()["T"]
    del c
    for p, (s, t) in enumerate([(1, 0), (4, 3)]):
        one = lcr.Cycle([clouds[s], clouds[t]], [(0, 1)], **kw)
        one.run()
        np.testing.assert_array_equal(one.results()["T"][0], T[p])


def test_default_radius_spans_no_near_mask(lcr):
    """The radius that the parameters default to, sqrt(DBL_MAX), spans more cells
    than an int counts: no near mask is built for it, and a pair gets the bits of a
    radius far beyond every distance."""
    cyc = synth.turntable_cycle(7, n_captures=2, yaw_step_deg=10.0, scale=1.0,
                                centre=(0.0, 0.0, -0.8))
    clouds = [c[:2000] for c in cyc.clouds]
    res = []
    for r in (1000.0, 1.3407807929942596e154):
        print_case(test="default_radius", r=r)
        c = lcr.Cycle(clouds, [(0, 1)], point_to_plane=False, max_corr_dist=r, max_iterations=6)
        c.run()
        res.append(c.results())
        del c
    for k in ("T", "iterations", "fitness"):
        np.testing.assert_array_equal(res[1][k], res[0][k])
