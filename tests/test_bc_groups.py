"""The grouping of boundary ranges into launches (csrc/update.hip group_bcs),
on the CPU: ranges of one group run at the same time, so none may write a
point that another reads or writes, and ranges that meet have to stay in
their order.  Checked point by point on random partitions of a block's faces,
with patches that share end points, overlap, or lie inside the block."""
import os
import random
import subprocess

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "openstc-dev_amd")

# reads "g n" and n lines "face dir rs[3] re[3]"; prints the ranges of a group per line
DRIVER = r"""
#include <cstdio>
#include <vector>
#include "flux_kernels.h"
int main() {
  int g, n;
  while (scanf("%d %d", &g, &n) == 2) {
    std::vector<ostc::BCDesc> b(n);
    for (int i = 0; i < n; ++i) {
      b[i].type = i;
      if (scanf("%d %d", &b[i].face, &b[i].dir) != 2) return 1;
      for (int &v : b[i].rs) if (scanf("%d", &v) != 1) return 1;
      for (int &v : b[i].re) if (scanf("%d", &v) != 1) return 1;
    }
    for (auto &group : ostc::group_bcs(b, g)) {
      for (auto &d : group) printf("%d ", d.type);
      printf("\n");
    }
    printf("end\n");
  }
}
"""


@pytest.fixture(scope="module")
def group(tmp_path_factory):
    root = tmp_path_factory.mktemp("groups")
    src, exe = root / "driver.cpp", root / "driver"
    src.write_text(DRIVER)
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "-std=c++17", "-O1", "-w", "-I",
                    os.path.join(PKG, "csrc"), str(src), "-o", str(exe), "-L" + PKG,
                    "-l:libostc.so", "-Wl,-rpath," + PKG], check=True, timeout=120)

    def run(g, ranges):
        text = "%d %d\n" % (g, len(ranges))
        text += "".join("%d %d %d %d %d %d %d %d\n" % ((f, d) + tuple(rs) + tuple(re)) for f, d, rs, re in ranges)
        out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True, timeout=60).stdout
        return [[int(v) for v in ln.split()] for ln in out.splitlines() if ln != "end"]

    return run


def _points(r, g, side):
    """The face layer and g layers outwards (side 1) or inwards (-1)."""
    face, direction, rs, re = r
    lo, hi = list(rs), list(re)
    if side * direction > 0:
        hi[face] += g
    else:
        lo[face] -= g
    return {(i, j, k) for i in range(lo[0], hi[0] + 1) for j in range(lo[1], hi[1] + 1)
            for k in range(lo[2], hi[2] + 1)}


def _check(groups, ranges, g):
    assert sorted(i for q in groups for i in q) == list(range(len(ranges)))
    level = {i: n for n, q in enumerate(groups) for i in q}
    wr = [_points(r, g, 1) for r in ranges]
    rd = [_points(r, g, -1) for r in ranges]
    for j in range(len(ranges)):
        for i in range(j):
            if wr[i] & wr[j] or wr[i] & rd[j] or rd[i] & wr[j]:
                assert level[i] < level[j], (ranges[i], ranges[j])
    assert all(q == sorted(q) for q in groups)


def _random_ranges(rng, m, g, dim):
    """Ranges as the block's set-up registers them: patches of its faces, most
    of them widened by the g ghosts along the face (walls are not), some on a
    layer inside the block."""
    out = []
    for _ in range(rng.randint(2, 9)):
        face = rng.randrange(dim)
        at = rng.choice((0, m[face] - 1, m[face] - 1 if rng.random() < 0.7 else rng.randrange(1, m[face])))
        wide = 0 if rng.random() < 0.3 else g
        rs, re = [0, 0, 0], [0, 0, 0]
        for d in range(3):
            if d == face:
                rs[d] = re[d] = at
            elif d >= dim:
                rs[d], re[d] = -g, g
            else:
                a, b = sorted((rng.randrange(m[d]), rng.randrange(m[d]))) if rng.random() < 0.6 else (0, m[d] - 1)
                rs[d], re[d] = a - wide, b + wide
        out.append((face, -1 if at == 0 else 1, rs, re))
    return out


@pytest.mark.parametrize("dim,g", [(2, 2), (2, 3), (3, 2)])
def test_groups_never_meet(group, dim, g):
    rng = random.Random(11 * dim + g)
    several = 0
    for _ in range(40):
        m = [rng.randint(4, 14), rng.randint(4, 14), rng.randint(4, 9) if dim == 3 else 1]
        ranges = _random_ranges(rng, m, g, dim)
        groups = group(g, ranges)
        _check(groups, ranges, g)
        several += any(len(q) > 1 for q in groups)
    assert several > 10  # the ranges do share launches


def test_check_sees_a_conflict():
    """The check itself: neighbouring walls that share a corner may not share a group."""
    a = (1, -1, [0, 0, 0], [9, 0, 0])
    b = (0, -1, [0, 0, 0], [0, 9, 0])
    _check([[0], [1]], [a, b], 2)
    with pytest.raises(AssertionError):
        _check([[0, 1]], [a, b], 2)
    with pytest.raises(AssertionError):
        _check([[1], [0]], [a, b], 2)
