"""CPU tier: the token tile and K split that the GEMM plans (mia_gemm_plan.h, compiled for the
host) for the shapes by which the GPU tests mean to reach each of its kernels on 256 CUs.  Retuned
costs that move a shape to another tile fail here."""

import ctypes
import os
import shutil
import subprocess

import pytest

import _gemm_shapes as GS

HERE = os.path.dirname(os.path.abspath(__file__))
# (enum in mia_kernels.h)
Q40_TILE, Q40, Q4K, F16, F16X2, Q6K = range(6)
SOURCES = {"q4_0": (Q40, Q40_TILE), "q4_k": (Q4K, F16), "f16": (F16,), "q6_k": (Q6K, F16X2),
           "f32": (F16X2,)}


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    so = tmp_path_factory.mktemp("plan") / "gemm_plan.so"
    subprocess.run([hipcc, "-O1", "-std=c++17", "-shared", "-fPIC", "--offload-arch=gfx950",
                    "--offload-host-only", "-x", "hip", os.path.join(HERE, "plan", "gemm_plan.cpp"),
                    "-o", str(so)], check=True, capture_output=True)
    lib = ctypes.CDLL(str(so))

    def f(src, S, N, K, plain=False, num_cus=256):
        tm, ks = ctypes.c_int(), ctypes.c_int()
        lib.plan(src, N, K, S, num_cus, int(plain), ctypes.byref(tm), ctypes.byref(ks))
        return tm.value, ks.value

    return f


@pytest.mark.parametrize("kind,S,N,K,split", GS.WIDE_GEMM)
def test_wide_gemm_shapes(plan, kind, S, N, K, split):
    # 128-token tiles whose last tile and last weight rows are ragged; the packed
    # form takes the same tile and split
    assert S % 128 and N % 256
    for src in SOURCES[kind]:
        tm, ks = plan(src, S, N, K)
        assert tm == 4 and (ks > 1) == split


@pytest.mark.parametrize("S,dim,hidden,split", GS.WIDE_LAYERS)
def test_wide_layer_shapes(plan, S, dim, hidden, split):
    # the fused gate / up launch of a Q4_K layer, from the file's blocks or packed
    assert S % 128
    for src in SOURCES["q4_k"]:
        tm, ks = plan(src, S, 2 * hidden, dim)
        assert tm == 4 and (ks > 1) == split


def test_split_of_many_tokens(plan):
    # the shape by which the GPU tests have a K split of more than 65,535 tokens
    S, N, K = GS.MANY_TOKENS
    assert S > 65535 and plan(Q6K, S, N, K)[1] > 1


@pytest.mark.parametrize("src,S,N,K,slow", [
    # choices that had cost 13 to 40 % more than another: a last round of a few
    # workgroups, and splits of weights that memory bounds
    (Q40_TILE, 777, 4096, 4096, (1, 2)), (Q4K, 777, 14336, 4096, (4, 2)),
    (F16, 777, 6144, 4096, (4, 4)), (F16X2, 33, 14336, 4096, (2, 4)),
    (F16X2, 300, 4096, 4096, (2, 8)), (Q4K, 64, 4096, 4096, (2, 16)),
])
def test_plan_avoids_slow_choices(plan, src, S, N, K, slow):
    assert plan(src, S, N, K) != slow


@pytest.mark.parametrize("kind", ["q4_0", "q4_k", "q6_k"])
def test_split_is_the_same_in_both_forms(plan, kind):
    a, b = SOURCES[kind]
    for N, K in ((4096, 4096), (14336, 4096), (4096, 14336), (1024, 4096), (520, 2048), (96, 512)):
        for S in (1, 8, 33, 64, 65, 100, 129, 300, 444, 512, 777, 1024, 2048, 5000):
            assert plan(a, S, N, K)[1] == plan(b, S, N, K)[1]
