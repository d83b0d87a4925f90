"""The library's choice of kernel for a matrix product (csrc/sh_gemm_plan.hpp), asked of the header
itself: it is host code, compiled here into a small program."""
import functools
import os
import subprocess
import tempfile
from collections import namedtuple

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
KINDS = ("pipe32", "ring128x256", "ring128x128", "ring64x128", "ring64x64", "ring32x64")
Plan = namedtuple("Plan", "kind ranges kc run one_plane_ok few")

SOURCE = r"""
#include "sh_gemm_plan.hpp"
#include <stdio.h>
int main() {
    int m, n, k, one, bf;
    while (scanf("%d %d %d %d %d", &m, &n, &k, &one, &bf) == 5) {
        const sh::GemmPlan p = sh::gemm_plan(m, n, k, one, bf);
        printf("%d %d %d %d %d %d\n", p.kind, p.ranges, p.kc, p.run, sh::gemm_one_plane(m, n, k), sh::linear_few(m, n, k, false));
    }
}
"""


@functools.lru_cache(None)
def _program():
    d = tempfile.TemporaryDirectory(prefix="gemm_plan")
    src = os.path.join(d.name, "main.cpp")
    with open(src, "w") as f:
        f.write(SOURCE)
    exe = os.path.join(d.name, "main")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "ane-training-experiments_amd", "csrc"),
                           src, "-o", exe])
    return exe, d


def plans(products):
    """Plan of each (M, N, K, one_plane[, bf16])."""
    text = "\n".join("%d %d %d %d %d" % (*p, 0)[:5] for p in products)
    out = subprocess.run([_program()[0]], input=text, capture_output=True, text=True, check=True).stdout
    rows = [[int(v) for v in line.split()] for line in out.splitlines()]
    assert len(rows) == len(products)
    return [Plan(KINDS[r[0]], *r[1:4], bool(r[4]), bool(r[5])) for r in rows]


def conv_kernel(s, in_dim, out_dim):
    """The kernel of a ConvEval: "few", or the plan's kind with its K ranges."""
    p = plans([(s, out_dim, in_dim, 0)])[0]
    return "few" if p.few else "%s/%d%s" % (p.kind, p.ranges, " in runs" if p.run else "")
