"""bench.py's split of its steps into graphs: every step once, in rotation
order, as long as asked for whatever --steps and --warmup are."""
import pytest

import bench


@pytest.mark.parametrize("steps,most,rotate", [(20, 32, 32), (5, 32, 32), (64, 32, 32), (100, 32, 32), (7, 1, 4),
                                               (50, 12, 8), (0, 32, 32), (33, 32, 16)])
def test_step_pieces(steps, most, rotate):
    pieces = bench.step_pieces(steps, most, rotate)
    layers = [l % rotate for first, count in pieces for l in range(first, first + count)]
    assert layers == [s % rotate for s in range(steps)]
    assert all(1 <= count <= most for _, count in pieces)
    assert all(count == most for _, count in pieces[:-1])  # one shorter piece at most
