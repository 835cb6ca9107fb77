"""What a call runs as, asked of the library's own choice without a GPU (nk_hip_planned_tile)."""
import random
import time

import pytest

from tests.support import STRIPS, route_of

COMPUTE_UNITS = 256  # what the library takes where it cannot ask a device


def strips_of(m, n, stages=2, config=STRIPS):
    return route_of("i8", "dots", m, n, 128 * stages, config)


def walked(m, n, rows, strip_tiles):
    """Tiles that the rounds of resident workgroups walk, one for starting and ending each strip included."""
    strips = -(-(-(-n // 256)) // strip_tiles)
    return -(-(-(-m // rows) * strips) // COMPUTE_UNITS) * (strip_tiles + 1)


# The number of strips against every other number that there is, rows of 128 (2 stages) and of 64 (8).
def test_no_number_of_strips_walks_less():
    rng = random.Random(3)
    for _ in range(300):
        stages = rng.choice((2, 8))
        m, n = int(10 ** rng.uniform(1.9, 5)), int(10 ** rng.uniform(2.2, 5.5))
        rows, route = 128 if stages == 2 else 64, strips_of(m, n, stages)
        assert route.shape == STRIPS and 1 <= route.strip_tiles <= -(-n // 256)
        assert route.units == -(-m // rows) * -(-(-(-n // 256)) // route.strip_tiles)
        tiles = -(-n // 256)
        least = min(walked(m, n, rows, length) for length in range(1, tiles + 1))
        assert walked(m, n, rows, route.strip_tiles) <= 1.06 * least, (m, n, stages) # (of the numbers the eight candidates leave out)


# Planning is part of the call: one with few rows took 2.8 us for it, more than some of them gain from the strips.
def test_planning_takes_no_time():
    def least(shape, config):
        best = 1e9
        for _ in range(30):
            begin = time.perf_counter()
            for _ in range(20):
                route_of("i8", "dots", *shape, config)
            best = min(best, (time.perf_counter() - begin) / 20)
        return best

    tiles, strips = least((100, 300_001, 256), 4), least((100, 300_001, 256), STRIPS)
    assert strips < tiles + 1.0e-6, f"{(strips - tiles) * 1e6:.2f} us more than for a fixed tile"
