"""Where the workgroups of a streaming prefill run (csrc/prefill_parts.h, prefill_common.h), compiled for the host: every workgroup of
every head group has exactly one place in the grid, in each of the orders; and which launches share KV heads as pairs, a head per
workgroup, or spread over the XCDs, on either side of the lines."""

import os
import subprocess
import textwrap

import pytest

import __graft_entry__ as entry

PROGRAM = textwrap.dedent(
    r"""
    #include <cstdio>
    #include <vector>
    #include "prefill_parts.h"
    using namespace ttpa;

    static PrefillArgs pass(int batch, int hq, int hkv, int sq, long keys, bool paged) {
      static const int32_t table = 0;
      PrefillArgs a = {};
      a.batch = batch, a.hq = hq, a.hkv = hkv, a.sq = sq, a.keys_bound = keys, a.keys_known = 1, a.cus = 256;
      a.pt = paged ? &table : nullptr;
      return a;
    }
    // every (group, rank) once, nothing else
    static int places(PrefillArgs a, int heads, int spg, bool spread) {
      const int grid = lay_out(a, heads, spg, spread), groups = a.batch * (a.hq / heads);
      std::vector<int> seen(groups * a.spg);
      int bad = grid % 8 != 0;
      for (int wg = 0; wg < grid; ++wg) {
        int y, rank;
        if (!workgroup_place(a, wg, y, rank)) continue;
        if (y < 0 || y >= groups || rank < 0 || rank >= a.spg || seen[y * a.spg + rank]++) return 1;
      }
      for (int n : seen) bad |= n != 1;
      return bad;
    }
    int main(int argc, char **argv) {
      for (int heads : {1, 2, 4, 5})
        for (int groups = 1; groups <= 35; ++groups)
          for (int sq : {1, 32, 33, 128, 300, 1000})
            for (int spg : {0, 1, 3})
              for (int spread = 0; spread < 2; ++spread)
                if (places(pass(groups, heads, 1, sq, sq, true), heads, spg, spread)) return printf("places %d %d %d %d %d\n", heads, groups, sq, spg, spread), 1;
      int v[6];
      while (scanf("%d %d %d %d %d %d", v, v + 1, v + 2, v + 3, v + 4, v + 5) == 6) {
        PrefillArgs a = pass(v[0], v[1], v[2], v[3], v[4] + v[3], true);
        const int heads = head_group_size(a, v[5]);
        set_parts(a, heads, stream_split(v[5]));
        printf("%d %d\n", heads, (int)spreads_groups(a, heads, v[5]));
      }
      return 0;
    }
    """
)

LINES = [
    # batch, query heads, KV heads, rows, tokens behind, head size -> heads per group, spread
    ((1, 40, 8, 224, 1216, 128), (5, 1)), ((1, 40, 8, 288, 2432, 128), (5, 1)), ((1, 40, 8, 384, 1600, 128), (5, 1)), ((1, 40, 8, 384, 2176, 128), (5, 1)), ((1, 40, 8, 384, 2432, 128), (5, 0)), ((1, 20, 4, 256, 2432, 128), (5, 1)),
    ((1, 28, 4, 256, 1216, 128), (7, 1)), ((1, 12, 4, 256, 1216, 256), (3, 1)),
    ((1, 40, 8, 128, 832, 128), (5, 0)), ((1, 40, 8, 192, 5504, 128), (5, 0)), ((1, 40, 8, 2048, 1216, 128), (5, 0)), ((1, 40, 8, 256, 1216, 64), (5, 0)),
    # one row block
    ((1, 40, 8, 32, 512, 128), (1, 0)), ((1, 40, 8, 32, 832, 128), (1, 0)), ((2, 40, 8, 32, 512, 128), (1, 0)), ((1, 10, 2, 17, 512, 64), (1, 0)),
    ((1, 40, 8, 32, 256, 128), (5, 0)), ((1, 40, 8, 32, 2432, 128), (5, 0)), ((2, 40, 8, 32, 640, 128), (5, 0)), ((3, 40, 8, 32, 512, 128), (5, 0)),
    ((1, 12, 2, 32, 512, 128), (2, 0)), ((6, 40, 8, 33, 512, 128), (5, 0)),
    # a multiple of four, and of one or two: one way only
    ((1, 32, 8, 32, 832, 128), (4, 0)), ((1, 32, 8, 256, 1216, 128), (4, 0)), ((1, 16, 8, 256, 1216, 128), (2, 0)), ((1, 16, 16, 256, 1216, 128), (1, 0)),
]


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    where = tmp_path_factory.mktemp("places")
    source, binary = where / "places.hip", where / "places"
    source.write_text(PROGRAM)
    csrc = os.path.join(entry.PKG_ROOT, "csrc")
    # (the host's code only: `quotient` and the placement are compiled for both sides)
    subprocess.run(["/opt/rocm/bin/hipcc", "-O1", "-std=c++17", "--offload-host-only", "-w", f"-I{csrc}", f"-I{entry.ROOT}/include", str(source), "-o", str(binary)],
                   check=True, capture_output=True, text=True)
    return str(binary)


def test_places_and_lines(program):
    asked = "\n".join(" ".join(map(str, case)) for case, _ in LINES)
    done = subprocess.run([program], input=asked, capture_output=True, text=True)
    assert done.returncode == 0, done.stdout
    got = [tuple(map(int, line.split())) for line in done.stdout.splitlines()]
    wrong = [(case, want, have) for (case, want), have in zip(LINES, got) if want != have]
    assert len(got) == len(LINES) and not wrong, wrong
