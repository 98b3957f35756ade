"""CPU checks of which kernel the shapes of the GPU tests take
(tests/cpp/route_query.cpp asks infer_amd/csrc/iq_plan.h, as the launchers
do), on 256 compute units and with a stream's workspace: a changed constant
must not quietly take a test away from the kernel that it is written for."""
import os
import subprocess

import pytest

from tests import test_gpu_gemm_paths as gemm_paths
from tests import test_gpu_rows_paths as rows_paths

HERE = os.path.dirname(os.path.abspath(__file__))
CUS, STREAM, STATIC = 256, 16 << 20, 4 << 20


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("routes") / "route_query")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-o", exe, os.path.join(HERE, "cpp", "route_query.cpp")],
                   check=True)

    def run(query):
        r = subprocess.run([exe], input=query + "\n", capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stdout
        return r.stdout.strip()

    return run


def gemm(ask, T, N, K, kind, x):
    return ask(f"gemm {T} {N} {K} {kind} {x} {CUS} {STREAM}")


def rows(ask, M, Ns, K, kind, part=STREAM):
    return ask(f"rows {M} {sum((n + 15) // 16 for n in Ns)} {K} {kind} {CUS} {part}")


def test_wide_tiles_shapes(ask):
    """Each of the wide-tile test's matrices takes wide tiles for at least
    one activation type, and together they cover both kinds of each tile."""
    seen = set()
    for N, K, Ts in gemm_paths.WIDE:
        here = set()
        for T in Ts:
            for kind in (0, 1):
                for x in ("fp32", "bf16"):
                    r = gemm(ask, T, N, K, kind, x)
                    if r.startswith("wide"):
                        here.add((kind, x, r.split()[1]))
        assert here, (N, K)
        seen |= here
    assert {(k, "bf16", "bm=256") for k in (0, 1)} | {(k, "fp32", "bm=128") for k in (0, 1)} <= seen


def test_last_row_blocks_shapes(ask):
    N, K, Ts = gemm_paths.LAST_BLOCKS
    for x in ("fp32", "bf16"):
        for kind in (0, 1):
            live = set()
            for T in Ts:
                r = gemm(ask, T, N, K, kind, x).split()
                assert r[0] == "wide", (T, kind, x)
                if r[1] == "bm=128":
                    live.add(r[-1])
            assert {f"live={v}" for v in ("1,0", "2,0", "3,0", "4,1", "4,2", "4,3")} <= live, (kind, x, live)


def test_non_finite_shapes(ask):
    for kind in (0, 1):
        bm = set()
        for N, K, T in gemm_paths.NON_FINITE:
            assert gemm(ask, T, N, K, kind, "fp32").startswith("wide")
            bm.update(gemm(ask, T, N, K, kind, "bf16").split()[1:2])
        assert {"bm=128", "bm=256"} <= bm


def test_rows_shapes(ask):
    for kind in (0, 1):
        for M in (5, 8, 9, 16, 17, 32):
            for Ns, K in rows_paths.MANY + (rows_paths.LONG if M <= 16 else []):
                assert rows(ask, M, Ns, K, kind).startswith("gemvw"), (kind, M, Ns, K)
        for Ns, K in rows_paths.SOME:
            assert any(rows(ask, M, Ns, K, kind).startswith("gemvw") for M in (9, 16, 17, 32)), (kind, Ns, K)
        # the non-finite rows, and odd group counts
        for M in (5, 16, 32):
            assert rows(ask, M, (1600,), 16384, kind).startswith("gemvw")
        for K in (1152, 3456, 19072):
            assert rows(ask, 12, (65541,), K, kind) == "other preferred"


def test_small_scratch_shapes(ask):
    s = rows_paths.SCRATCH
    assert rows(ask, s["M"], (s["inside"],), s["K"], 1, STATIC).startswith("gemvw")
    assert rows(ask, s["M"], (s["beyond"],), s["K"], 1, STATIC) == "other room"
