"""Pieces of camera segments (host): they partition the segment's parameters, and wherever the camera
stands the scene is shared among many of them."""
import numpy as np
import pytest

from gpuupbp_amd import capi


def _pieces(o, d, t0, t1, ball, piece_len):
    seg = np.array([*o, t0, *d, t1], np.float32)
    b = np.array(ball, np.float32)
    out = np.zeros((64, 4), np.float32)
    n = capi.lib().upbp_test_pieces(seg.ctypes.data, b.ctypes.data, piece_len, out.ctypes.data, 64)
    assert 1 <= n <= 32
    return out[:n].astype(np.float64)


def _partition(p, t0, t1):
    assert p[0, 0] <= -1e36 * 0.99 and p[-1, 1] >= 1e36 * 0.99
    assert np.array_equal(p[1:, 0], p[:-1, 1])  # [lo, hi) of neighbours meet
    assert p[0, 2] == np.float32(t0) and p[-1, 3] == np.float32(t1)
    assert np.array_equal(p[1:, 2], p[1:, 0]) and np.array_equal(p[:-1, 3], p[:-1, 1])
    assert (np.diff(p[:, 2]) >= 0).all()


@pytest.mark.parametrize("away", [0.0, 1.5, 3.0, 20.0, 300.0])
@pytest.mark.parametrize("end", [2.0, 60.0, 1e4, 1e36])
@pytest.mark.parametrize("offset", [0.0, 0.9])
def test_the_scene_is_in_many_pieces_from_any_distance(away, end, offset):
    radius, c = 1.7, np.array([0.3, -0.2, 5.0])
    d = np.array([0.6, 0.0, 0.8])
    side = np.array([0.0, 1.0, 0.0])
    o = c - away * radius * d + offset * radius * side
    p = _pieces(o, d, 0.01, end, [*c, 2 * radius], 0.05)
    _partition(p, 0.01, end)
    h = radius * np.sqrt(1 - offset ** 2)  # the scene's chord along the ray
    lo, hi = max(0.01, away * radius - h), min(end, away * radius + h)
    if hi > lo:
        share = (np.minimum(p[:, 3], hi) - np.maximum(p[:, 2], lo)) / (hi - lo)
        # the ball's chord is at most 2 sqrt((2 radius)^2 - offset^2) long and cut in 32 (or at 0.05):
        # a piece holds at most 4 radii / 32, or the piece length, of the scene
        assert share.max() <= max(4 * radius / 32, 0.05) / (hi - lo) * 1.01 + 1e-3, share.max()


def test_a_segment_outside_the_ball_is_one_piece():
    for o, d, t0, t1 in (((0, 9, 0), (1, 0, 0), 0.0, 50.0), ((20, 0, 0), (1, 0, 0), 0.0, 50.0),
                         ((-20, 0, 0), (1, 0, 0), 0.0, 5.0), ((-20, 0, 0), (1, 0, 0), 30.0, 1e36)):
        p = _pieces(o, d, t0, t1, [0, 0, 0, 3], 0.1)
        assert len(p) == 1
        _partition(p, t0, t1)


def test_without_a_scene_radius_the_whole_segment_is_cut():
    p = _pieces((5, 0, 0), (0, 1, 0), 1.0, 9.0, [0, 0, 0, 1e36], 1.0)
    assert len(p) == 8
    _partition(p, 1.0, 9.0)
    assert np.allclose(np.diff(p[:, 2]), 1.0)


def test_no_piece_length_is_one_piece():
    assert len(_pieces((0, 0, 0), (0, 1, 0), 0.0, 9.0, [0, 0, 0, 3], 0.0)) == 1
