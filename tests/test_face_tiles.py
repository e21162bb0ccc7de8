"""Assignment of the faces' tiles to the workgroups of the one launch that covers three directions."""
import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "opencfd-ec_amd" / "csrc"
GROUP = int(re.search(r"constexpr int FACE_GROUP = (\d+);", (CSRC / "ocfd_dev.h").read_text()).group(1))


def face_grid(n):
    return 8 * 3 * GROUP * (((max(n) + 7) // 8 + GROUP - 1) // GROUP)


def face_tile(w, n):
    xcd, e = w % 8, w // 8
    d = e // GROUP % 3
    u, per = e // (3 * GROUP) * GROUP + e % GROUP, (n[d] + 7) // 8
    t = xcd * per + u
    return (d, t) if u < per and t < n[d] else None


@pytest.mark.parametrize("n", [(1, 1, 1), (7, 8, 9), (8, 7, 6), (127, 128, 129), (8 * GROUP, 8 * GROUP + 1, 8 * GROUP - 1),
                               (1000, 517, 3), (3, 4099, 2048), (0, 0, 0), (5, 0, 17)])
def test_each_tile_of_each_direction_in_one_workgroup(n):
    got = sorted(x for x in (face_tile(w, n) for w in range(face_grid(n))) if x)
    assert got == [(d, t) for d in range(3) for t in range(n[d])]
