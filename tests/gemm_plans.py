"""The launch plan of the f16 GEMMs (csrc/gemm_plan.hpp), evaluated by the host compiler."""
import os
import shutil
import subprocess
import tempfile

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "slang_amd", "csrc")
PROGRAM = r"""
#include <cstdio>
#include "gemm_plan.hpp"
using namespace g4a;
int main() {
    int ws, M, K, n, rows[3];
    while (scanf("%d %d %d %d", &ws, &M, &K, &n) == 4) {
        for (int i = 0; i < n; ++i)
            if (scanf("%d", rows + i) != 1) return 1;
        const SplitRoom room = split_room(M, K, n, rows);
        const GemmPlan p = gemm_plan(M, K, n, rows, ws ? room.max_splits : 1);
        const TileCfg& t = kTiles[p.cfg];
        printf("%d %d %d %d %d %d %zu\n", p.cfg, p.tiles, p.splits, t.bm, t.bn, t.step2 > 0.0f, room.ws_bytes);
    }
}
"""


def plans(shapes):
    """shapes: (workspace, M, K, weight rows of each matrix (2 n for the gate/up pair)). Returns for
    each a dict of cfg, tiles, splits, bm, bn, shared (two workgroups a CU), ws_bytes; None without
    a host compiler."""
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        return None
    with tempfile.TemporaryDirectory() as d:
        src, exe = os.path.join(d, "plan.cpp"), os.path.join(d, "plan")
        with open(src, "w") as f:
            f.write(PROGRAM)
        subprocess.run([cxx, "-std=c++17", "-O1", f"-I{CSRC}", src, "-o", exe], check=True, capture_output=True, text=True)
        lines = "".join(f"{int(ws)} {M} {K} {len(rows)} {' '.join(map(str, rows))}\n" for ws, M, K, rows in shapes)
        out = subprocess.run([exe], input=lines, capture_output=True, text=True, check=True).stdout.split("\n")
    keys = ("cfg", "tiles", "splits", "bm", "bn", "shared", "ws_bytes")
    return [dict(zip(keys, map(int, line.split()))) for line in out if line]
