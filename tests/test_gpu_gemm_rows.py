"""Stored GEMMs of row-major A at more than 16 rows (K-split blocks, 64 x 128 ring blocks) against
the one-tile kernel run on 16 rows at a time: every GEMM sums an output's 256-wide k-block chains
in k-block order whatever the other rows are, so the bits must be equal; and against float64
within one bf16 rounding plus K f32 roundings of the terms' magnitudes."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    from qwen35 import Engine
    e = Engine(max_rows=64, max_ctx=64, seed=None)
    yield e
    e.close()


# sizes at the edges of the 32-row / 64-row blocks, of the 16 / 32 / 128-column blocks, of one
# and two rounds of 256 blocks (where the forms change) and of 1 .. 16 k-blocks
@pytest.mark.parametrize("N,K,M,pad", [
    (1024, 3584, 17, 0), (1024, 3584, 33, 8), (1024, 3584, 128, 0), (1024, 3584, 129, 0), (1024, 3584, 511, 0),
    (1024, 3584, 512, 0), (1024, 3584, 513, 0), (1024, 2048, 257, 0), (1024, 2048, 1999, 16), (1040, 3584, 700, 0),
    (16, 4096, 40, 0), (48, 4096, 31, 0), (272, 1280, 65, 0), (1024, 256, 100, 0), (1024, 256, 900, 0),
    (1008, 512, 1100, 8), (4112, 768, 300, 0), (2048, 2304, 1000, 0),
    # K = 1024: either side of the line between the 32 x 64 and the 64 x 128 blocks (153 of 256)
    (5120, 1024, 192, 0), (5120, 1024, 256, 8), (7168, 1024, 449, 0), (8224, 1024, 384, 0), (2064, 1024, 600, 0), (128, 1024, 2048, 0)])
def test_row_major_gemm_equals_one_tile_kernel(eng, N, K, M, pad):
    import torch
    print(f"rows gemm N={N} K={K} M={M} ldx={K + pad}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(N + K + M)
    W = (0.02 * torch.randn(N, K, generator=g, device="cuda")).to(torch.bfloat16)
    buf = torch.randn(M, K + pad, generator=g, device="cuda").to(torch.bfloat16)
    X = buf[:, :K]
    Wt = torch.empty_like(W)
    Y = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device="cuda")      # a guard row after the last
    Z = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    torch.cuda.synchronize()   # torch-stream inputs complete before the engine stream reads them
    eng.op_tile_weight(W.data_ptr(), N, K, Wt.data_ptr())
    eng.op_gemm_a(Wt.data_ptr(), N, K, 0, X.data_ptr(), K + pad, 0, 0, 0, M, Y.data_ptr())
    for r in range(0, M, 16):
        eng.op_gemm_a(Wt.data_ptr(), N, K, 0, X[r:].data_ptr(), K + pad, 0, 0, 0, min(16, M - r), Z[r:].data_ptr())
    eng.sync()
    assert torch.equal(Y[:M].view(torch.int16), Z.view(torch.int16))
    assert (Y[M] == 7.0).all()
    ref = X.double() @ W.double().t()
    ulp = ref.abs().clamp_min(1e-30).log2().floor().sub(7).exp2()
    acc = (X.double().abs() @ W.double().abs().t()) * (K * 2.0 ** -24)
    assert ((Y[:M].double() - ref).abs() <= ulp + acc).all()


@pytest.mark.parametrize("F,M", [(3584, 256), (3584, 193), (1232, 500), (3584, 1100)])
def test_row_major_swiglu_equals_pipelined_form(eng, F, M):
    """The SwiGLU epilogue from row-major A in 64 x 128 blocks against the k-block-pipelined GEMM
    (option gemm_pre 0), bit for bit; F = 1232 ends inside a block's gate tiles."""
    import torch
    from qwen35 import Engine
    print(f"rows swiglu F={F} M={M}", flush=True)
    e = Engine(max_rows=2048, max_ctx=64, seed=None)
    try:
        g = torch.Generator(device="cuda").manual_seed(F + M)
        W = (0.02 * torch.randn(2 * F, 1024, generator=g, device="cuda")).to(torch.bfloat16)
        X = torch.randn(M, 1024, generator=g, device="cuda").to(torch.bfloat16)
        Wt = torch.empty_like(W)
        Y = [torch.full((M + 1, F), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
        torch.cuda.synchronize()
        e.op_tile_weight(W.data_ptr(), 2 * F, 1024, Wt.data_ptr())
        for form, y in zip((1, 0), Y):
            e.set_option("gemm_pre", form)
            e.op_gemm_a(Wt.data_ptr(), 2 * F, 1024, 5, X.data_ptr(), 1024, 0, 0, 0, M, y.data_ptr())
        e.sync()
        assert torch.equal(Y[0].view(torch.int16), Y[1].view(torch.int16))
        assert (Y[0][M] == 7.0).all()
    finally:
        e.close()
