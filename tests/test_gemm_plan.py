"""The prompt GEMM's launch shapes (gemm_plan.h, host arithmetic without HIP),
compiled alone and asked for every row count of a prompt block."""
import ctypes as C
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14
BLOCK = 512  # tokens of a prompt block

SHIM = """
#include "gemm_plan.h"
using namespace lrs;
extern "C" size_t work(uint32_t M, const uint32_t *N, const uint32_t *t, uint32_t n, uint32_t K, int prec) {
    return gemm_work_bytes(M, N, t, n, K, prec);
}
extern "C" uint32_t shape(uint32_t M, const uint32_t *N, const uint32_t *t, uint32_t n, uint32_t K, int prec) {
    const PgPlan p = pg_plan(M, N, t, n, K / 256, prec);
    return p.mt << 16 | p.ks;
}
extern "C" size_t most(uint32_t M, const uint32_t *N, const uint32_t *t, uint32_t n, uint32_t K, int prec) {
    return gemm_work_most(M, N, t, n, K, prec);
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(SHIM)
    so = d / "plan.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC",
                    "-I", os.path.join(REPO, "llama.rs_amd", "csrc"), str(d / "plan.cpp"), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))
    for f in (lib.work, lib.most):
        f.restype = C.c_size_t
    for f in (lib.work, lib.most, lib.shape):
        f.argtypes = [C.c_uint32, C.c_void_p, C.c_void_p, C.c_uint32, C.c_uint32, C.c_int]
    return lib


def args(ns, ts):
    u = C.c_uint32 * len(ns)
    return u(*ns), u(*ts), len(ns)


# (n_in, rows of each weight, types): the projections of the 32B and 14B dense
# and the 27B hybrid layers, gate / up and q / k / v as one launch
SETS = [(5120, (27648, 27648), (Q4_K, Q4_K)), (5120, (27648, 27648), (Q5_K, Q5_K)), (27648, (5120,), (Q6_K,)),
        (5120, (5120, 1024, 1024), (Q4_K, Q4_K, Q6_K)), (5120, (5120, 1024, 1024), (Q5_K, Q5_K, Q6_K)),
        (5120, (13824, 13824), (Q4_K, Q4_K)), (13824, (5120,), (Q6_K,)), (5120, (13824,), (Q8_0,)),
        (5120, (17408, 17408), (Q5_K, Q5_K)), (17408, (5120,), (Q6_K,)), (4096, (13824,), (Q4_K,)),
        (4096, (4096, 1024, 1024), (Q5_K, Q5_K, Q6_K)), (512, (512,), (Q4_K,))]


@pytest.mark.parametrize("k,ns,ts", SETS)
@pytest.mark.parametrize("prec", [1, 3])
def test_scratch_of_a_block_covers_every_shorter_one(plan, k, ns, ts, prec):
    """The buffer of a prompt block holds the partial sums of any number of
    tokens up to the block's (fewer tokens may take more slices)."""
    n, t, c = args(ns, ts)
    most = plan.most(BLOCK, n, t, c, k, prec)
    assert all(plan.work(m, n, t, c, k, prec) <= most for m in range(1, BLOCK + 1))


# bf16 Q4_K over 13824 x 5120: one row tile without a split takes 116 us at 384
# rows and 118 at 448, where four take 79 and 91
@pytest.mark.parametrize("m", [289, 320, 352, 378, 384, 385, 400, 416, 448, 512, 1024, 2048])
def test_bf16_q4_k_takes_several_row_tiles(plan, m):
    n, t, c = args((13824,), (Q4_K,))
    assert plan.shape(m, n, t, c, 5120, 1) >> 16 > 1


@pytest.mark.parametrize("k,ns,ts", SETS)
@pytest.mark.parametrize("prec", [1, 3])
@pytest.mark.parametrize("m", [1, 31, 32, 33, 64, 65, 512, 4096, 65535, 65536, 1 << 20])
def test_shapes_are_launchable(plan, k, ns, ts, prec, m):
    """Row tiles that the kernel is built for, not more slices than super-blocks,
    and none past the reduce's grid."""
    n, t, c = args(ns, ts)
    s = plan.shape(m, n, t, c, k, prec)
    mt, ks = s >> 16, s & 0xFFFF
    assert mt in ((1, 2) if prec == 3 else (1, 2, 4)) and 1 <= ks <= min(32, k // 256)
    assert m <= 65535 or ks == 1


# the edge that the prompt block tests on the GPU stand on either side of
@pytest.mark.parametrize("k,ns,ts,m", [(2048, (8448,), (Q6_K,), 128)])
def test_split_ends_where_the_block_tests_stand(plan, k, ns, ts, m):
    n, t, c = args(ns, ts)
    assert plan.shape(m, n, t, c, k, 3) & 0xFFFF > 1 and plan.shape(m + 1, n, t, c, k, 3) & 0xFFFF == 1
