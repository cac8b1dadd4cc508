"""GPU truncated distance field (rtr_tdf, rtr_tdf_points) against the
brute-force oracle of kernel.cu:9-31's semantics: bit-identical."""
import numpy as np
import pytest

import oracle
import realtime_robot_amd as R
from realtime_robot_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,n_occ,trunc2", [((30, 30, 30), 600, 900.0), ((64, 48, 40), 300, 900.0),
                                               ((7, 130, 3), 20, 50.0), ((1100, 3, 2), 5, 1e6),
                                               ((16, 16, 16), 0, 900.0)])
def test_tdf_matches_brute_force(dims, n_occ, trunc2):
    rng = np.random.default_rng(sum(dims) + n_occ)
    occ = rng.integers(-2, np.array(dims) + 2, size=(n_occ, 3)).astype(np.int32)   # some outside the grid
    got = R.tdf(occ, dims, trunc2)
    ref = oracle.tdf(occ, dims, trunc2)
    assert np.array_equal(got, ref)


def test_tdf_of_key_point_box_like_the_reference():
    """The reference's use: the occupied 1 cm voxels of a cloud inside a
    0.3 m box around a key point (key_point.h:287-308), 30^3 grid, cap 900."""
    src, tgt, _ = synth.config1_pair(0)
    center = tgt[1234].astype(np.float64)
    lo = (center - 0.15).astype(np.float32)
    got = R.tdf_points(tgt, lo, 0.01, (30, 30, 30), 900.0)
    f = (tgt - lo) * (np.float32(1.0) / np.float32(0.01))
    inside = np.all((f >= 0) & (f < 30), axis=1)
    occ = np.unique(f[inside].astype(np.int32), axis=0)
    ref = oracle.tdf(occ, (30, 30, 30), 900.0)
    assert len(occ) > 50 and np.array_equal(got, ref)


@pytest.mark.parametrize("dims", [(1, 1, 1), (2, 1, 3), (5, 4, 1), (6, 9, 13), (700, 1, 2), (1, 66, 1), (3, 2, 259)])
@pytest.mark.parametrize("cap", [0.25, 1.0, 30.5, 900.0, 1.0e9])
def test_outward_passes_match_brute_force(dims, cap):
    """Lines shorter than, as long as and just beyond the four offsets taken
    at a time, caps below one voxel, between whole numbers and out of reach,
    one voxel occupied, all of one face, and none."""
    rng = np.random.default_rng(sum(dims))
    d = np.array(dims)
    one = (rng.random((1, 3)) * d).astype(np.int32)
    face = np.stack([np.zeros(8, np.int32), *(rng.integers(0, d[a], 8) for a in (1, 2))], 1).astype(np.int32)
    for occ in (one, face, np.zeros((0, 3), np.int32)):
        assert np.array_equal(R.tdf(occ, dims, cap), oracle.tdf(occ, dims, cap))


@pytest.mark.parametrize("dims", [(41, 43, 45), (300, 17, 16), (4096, 6, 3), (70, 61, 33), (4, 9, 4000), (4096, 33, 1),
                                  (1, 4096, 33), (129, 130, 11)])
@pytest.mark.parametrize("cap", [900.0, 1.0e9])
def test_passes_by_field_size_match_brute_force(dims, cap):
    """The passes change with the field's size (one voxel a lane and eight or
    sixteen offsets at once, or runs of four voxels): lines that end in every part
    of a run, shorter than one, and longer than the offsets ever go."""
    rng = np.random.default_rng(sum(dims))
    d = np.array(dims)
    few = (rng.random((3, 3)) * d).astype(np.int32)
    many = (rng.random((2000, 3)) * d).astype(np.int32)
    for occ in (few, many):
        assert np.array_equal(R.tdf(occ, dims, cap), oracle.tdf(occ, dims, cap))
