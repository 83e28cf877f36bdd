"""Shapes whose plan (tile, K split) on 256 CUs the GPU tests rely on; test_gemm_plan.py checks
the plans."""

# (weights, S, N, K, K split): 128-token tiles, ragged at both ends
WIDE_GEMM = [(kind, *shape) for kinds, shapes in (
    (("q4_k", "f16"), ((1100, 2056, 2048, True), (1100, 4104, 1024, False))),
    (("q6_k", "f32"), ((900, 1032, 2048, True), (1100, 4104, 512, False))),
) for kind in kinds for shape in shapes]

# (S, dim, hidden, K split of the fused gate / up GEMM): its 128-token tiles
WIDE_LAYERS = [(300, 1024, 8192, False), (300, 2048, 4096, True)]

# S, N, K of a Q6_K product
MANY_TOKENS = (66000, 32, 4096)
