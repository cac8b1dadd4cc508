"""The keypoint + TDF + yaw-search coarse proposer (rtr_coarse_*) against its
CPU restatement (oracle/coarse.py): keypoints and occupied voxels bit-exact,
keypoint-pair scores to float summation order, and the proposals it makes on
gravity-aligned pairs."""
import numpy as np
import pytest

from oracle import coarse as oc
from realtime_robot_amd import synth
from realtime_robot_amd.coarse import CoarseProposer

pytestmark = pytest.mark.gpu


def test_keypoints_occupancy_and_scores_match_oracle():
    srcs, tgts, _ = synth.config4_yaw_batch(2, seed_offset=300, ns_range=(3000, 9000), nt_range=(5000, 12000))
    cp = CoarseProposer()
    cp.set_clouds(srcs, tgts)
    sc, yaw, kp = cp.pair_scores()
    occ = cp.occupancy()
    for p in range(2):
        ref, ks, kt = oc.pair_scores(srcs[p], tgts[p])
        assert np.array_equal(kp[2 * p], ks) and np.array_equal(kp[2 * p + 1], kt)
        for j in range(oc.KEYS):
            assert np.array_equal(occ[p][j], oc.occupancy(srcs[p], ks[j]))
        best = ref.min(axis=2)
        rejected = best >= 1e38
        assert np.array_equal(sc[p] >= 1e38, rejected)
        ok = ~rejected
        rel = np.abs(sc[p][ok] - best[ok]) / np.maximum(best[ok], 1e-3)
        print(p, "pairs kept", ok.sum(), "max rel score error", rel.max())
        assert rel.max() < 1e-5
        # the best yaw agrees wherever the oracle's best is not a near-tie
        srt = np.sort(ref, axis=2)
        clear = ok & (srt[:, :, 1] - srt[:, :, 0] > 1e-3 * np.maximum(srt[:, :, 0], 1e-3))
        assert np.array_equal(yaw[p][clear], np.argmin(ref, axis=2)[clear])


def test_coarse_proposals_on_gravity_aligned_pairs():
    srcs, tgts, gts = synth.config4_yaw_batch(16, seed_offset=310, ns_range=(3000, 20000), nt_range=(10000, 60000))
    cp = CoarseProposer()
    cp.set_clouds(srcs, tgts)
    T, s = cp.propose()
    rot = [np.degrees(np.arccos(np.clip((np.trace(T[i][:3, :3].T @ gts[i][:3, :3]) - 1) / 2, -1, 1)))
           for i in range(16)]
    rmse = [synth.rmse_between(T[i], gts[i], srcs[i]) for i in range(16)]
    print("coarse: rotation error deg", np.round(rot, 1), "rmse m", np.round(rmse, 3), f"{cp.last_ms():.2f} ms")
    assert np.all(np.abs(np.linalg.det(T[:, :3, :3]) - 1) < 1e-9)
    assert np.mean(np.array(rot) < 15.0) >= 0.75


def test_ablation_learned_vs_reference_method():
    """The learned proposer against the reference's own coarse method and
    against no proposer, each followed by the same ICP refine: on full-SO(3)
    pairs the learned path registers more pairs than either; on gravity-
    aligned pairs the yaw search beats starting without a proposer."""
    from realtime_robot_amd import ablation
    out = ablation.run(pairs=24, seed_offset=500, verbose=False)
    for wl in ("so3", "yaw"):
        print(wl, {k: (v["within_1mm"], round(v["proposal_rot_err_deg_median"], 1)) for k, v in out[wl].items()})
    so3, yaw = out["so3"], out["yaw"]
    assert so3["learned"]["within_1mm"] > so3["coarse"]["within_1mm"]
    assert so3["learned"]["within_1mm"] > so3["none"]["within_1mm"]
    assert yaw["coarse"]["within_1mm"] > yaw["none"]["within_1mm"]


@pytest.mark.parametrize("res", [0.004, 0.01, 0.05, 2e18])
def test_scores_over_resolutions_match_oracle(res):
    """Field and lookups from nearly empty to full boxes, and a resolution
    whose arithmetic needs the range checks; clouds smaller than the keypoint
    count among them.  Sums of whole numbers: equal to float rounding of the mean."""
    rng = np.random.default_rng(8)
    srcs = [rng.uniform(-0.2, 0.2, (n, 3)).astype(np.float32) for n in (5, 900)]
    tgts = [rng.uniform(-0.2, 0.2, (n, 3)).astype(np.float32) for n in (700, 40)]
    cp = CoarseProposer()
    cp.set_clouds(srcs, tgts)
    sc, yaw, kp = cp.pair_scores(res)
    for p in range(2):
        ks, kt = oc.keypoints(srcs[p]), oc.keypoints(tgts[p])
        for i, j in ((0, 0), (1, 4), (3, 2), (31, 31)):
            grid, inner = oc.target_grid(tgts[p], kt[i], np.float32(res))
            ref = oc.score(oc.occupancy(srcs[p], ks[j], np.float32(res)), grid, inner, np.float32(res))
            if ref[0] >= 1e38:
                assert sc[p, i, j] >= 1e38
                continue
            assert abs(sc[p, i, j] - ref.min()) <= 1e-6 * max(ref.min(), 1e-3)
            assert ref[yaw[p, i, j]] <= ref.min() * (1 + 1e-6)


@pytest.mark.parametrize("m", [1, 3, 64, 513, 1024])
def test_device_selection_matches_host(m):
    """Candidates sorted and built on the device against the same choice from
    the pair scores on the host: the m best by (score, index), the lowest
    chamfer among them."""
    srcs, tgts, _ = synth.config4_yaw_batch(3, seed_offset=330, ns_range=(700, 3000), nt_range=(900, 4000))
    srcs[2], tgts[2] = srcs[2][:20], tgts[2][:300]
    cp = CoarseProposer()
    cp.set_clouds(srcs, tgts)
    T, s = cp.propose(candidates=m, tau=0.1)
    sc, yaw, kp = cp.pair_scores()
    for p in range(3):
        order = np.lexsort((np.arange(1024), sc[p].reshape(-1)))[:m]
        ang = yaw[p].reshape(-1)[order] * (2 * np.pi / 36)
        ki, kj = kp[2 * p + 1][order // 32].astype(np.float64), kp[2 * p][order % 32].astype(np.float64)
        c, sn = np.cos(ang), np.sin(ang)
        poses = np.zeros((m, 4, 4))
        poses[:, 0, 0], poses[:, 0, 1], poses[:, 1, 0], poses[:, 1, 1], poses[:, 2, 2], poses[:, 3, 3] = c, -sn, sn, c, 1, 1
        poses[:, 0, 3] = ki[:, 0] - (c * kj[:, 0] - sn * kj[:, 1])
        poses[:, 1, 3] = ki[:, 1] - (sn * kj[:, 0] + c * kj[:, 1])
        poses[:, 2, 3] = kp[2 * p + 1][order // 32, 2] - kp[2 * p][order % 32, 2]   # a float difference
        hit = np.where(np.abs(poses - T[p]).max(axis=(1, 2)) < 1e-12)[0]
        assert len(hit) >= 1
        a, b = oc.subsample(srcs[p], 1024).astype(np.float64), oc.subsample(tgts[p], 1024).astype(np.float64)
        chamfer = lambda P: np.mean(np.minimum(((a @ P[:3, :3].T + P[:3, 3])[:, None] - b[None]) ** 2 @ np.ones(3), 0.01).min(1))
        few = sorted(set(list(hit[:1]) + list(range(0, m, max(1, m // 24)))))
        best = {k: chamfer(poses[k]) for k in few}
        assert abs(s[p] - best[hit[0]]) < 1e-5 * max(s[p], 1e-4) + 1e-7
        assert all(v >= s[p] - 1e-6 for v in best.values())
