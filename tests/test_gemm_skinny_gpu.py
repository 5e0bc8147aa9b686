"""The GEMMs of few rows (M <= 48; up to K 4096 past 16 rows): the streaming kernel behind iron_gemm_bf16_nt,
iron_gemm_bf16_nn, iron_gemm_i4g32_nt and iron_gemm_bf16_nt_swiglu, at the edges of its row tiles, column tiles and
K units, against float64 and against each other (the forms share the split of K and the order of the sums)."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16

# row tiles of 16, 32 and 48 and their edges; K of one step, half and whole 128-deep units, fewer and more units than
# waves; N of one column, ragged, and past the two-column-tile rule (8192); K > 4096 only up to 16 rows
SHAPES = [(1, 64, 1), (1, 8256, 24), (15, 192, 40), (16, 1024, 130), (16, 4160, 64), (17, 128, 200), (31, 2048, 48),
          (32, 320, 8200), (33, 64, 16), (47, 1088, 520), (48, 4096, 72), (48, 640, 8208), (9, 576, 8197)]


def _inputs(gpu, M, K, N, signed=True):
    g = torch.Generator().manual_seed(M + 3 * K + 7 * N)
    A = torch.randn(M, K, generator=g).to(BF16)
    codes = torch.randint(0, 256, (N, K // 2), generator=g, dtype=torch.uint8)
    scales = (0.001 + 0.009 * torch.rand(N, K // 32, generator=g)).to(BF16)
    q = torch.stack([codes & 15, codes >> 4], 2).reshape(N, K).int()
    if signed:
        q = torch.where(q > 7, q - 16, q)
    W = (q.double() * scales.double().repeat_interleave(32, 1)).to(BF16)  # exact in 64 bits, one rounding
    return A.to(gpu), codes.to(gpu), scales.to(gpu), W.to(gpu)


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_skinny_forms(gpu, M, K, N):
    from iron_amd import _lib

    A, codes, scales, W = _inputs(gpu, M, K, N)
    s = _lib.stream_handle(gpu)
    assert _lib.query("iron_gemm_splitk_choose", M, N, K) == 1
    assert _lib.query("iron_gemm_i4g32_splitk_choose", M, N, K) == 1
    out = torch.full((M + 1, N), 7.0, dtype=BF16, device=gpu)
    _lib.call("iron_gemm_bf16_nt", A.data_ptr(), W.data_ptr(), out.data_ptr(), M, N, K, N, 0, 0, 0.0, 0.0, s)
    exact = A.double() @ W.double().t()
    torch.cuda.synchronize()
    assert (out[M] == 7.0).all()
    # a bf16 rounding (2^-9 of the value) on top of fp32 sums of K products (K 2^-24 of the sum of their magnitudes)
    bound = exact.abs() * 2.0**-8 + K * 2.0**-23 * (A.double().abs() @ W.double().abs().t())
    assert ((out[:M].double() - exact).abs() <= bound).all()

    for signed in (True, False):
        Ai, c, sc, Wi = (A, codes, scales, W) if signed else _inputs(gpu, M, K, N, signed=False)
        ref, got = torch.empty(M, N, dtype=BF16, device=gpu), torch.empty(M, N, dtype=BF16, device=gpu)
        _lib.call("iron_gemm_bf16_nt", Ai.data_ptr(), Wi.data_ptr(), ref.data_ptr(), M, N, K, N, 0, 0, 0.0, 0.0, s)
        _lib.call("iron_gemm_i4g32_nt", Ai.data_ptr(), c.data_ptr(), sc.data_ptr(), got.data_ptr(), M, N, K, N, 0, 0, 0.0,
                  0.0, int(signed), 1, None, 0, s)
        torch.cuda.synchronize()
        assert torch.equal(got, ref)
    if N % 8 == 0:
        B, got = W.t().contiguous(), torch.empty(M, N, dtype=BF16, device=gpu)
        _lib.call("iron_gemm_bf16_nn", A.data_ptr(), B.data_ptr(), got.data_ptr(), M, N, K, N, 0, 0, 0.0, 0.0, 1, None, 0, s)
        torch.cuda.synchronize()
        assert torch.equal(got, out[:M])


@pytest.mark.parametrize("M,K,F", [(1, 64, 64), (16, 8256, 128), (20, 1024, 320), (48, 448, 8192)])
def test_skinny_swiglu_pair(gpu, M, K, F):
    """The pair is bit-identical to its two halves followed by iron_silu_mul."""
    from iron_amd import _lib

    A, _, _, W = _inputs(gpu, M, K, 2 * F)
    s = _lib.stream_handle(gpu)
    pair = W.view(F // 64, 2, 64, K)
    halves = []
    for h in (0, 1):
        Wh, C = pair[:, h].reshape(F, K).contiguous(), torch.empty(M, F, dtype=BF16, device=gpu)
        _lib.call("iron_gemm_bf16_nt", A.data_ptr(), Wh.data_ptr(), C.data_ptr(), M, F, K, F, 0, 0, 0.0, 0.0, s)
        halves.append(C)
    ref = torch.empty(M, F, dtype=BF16, device=gpu)
    _lib.call("iron_silu_mul", halves[0].data_ptr(), halves[1].data_ptr(), ref.data_ptr(), M * F, s)
    H = torch.full((M, F + 64), 3.0, dtype=BF16, device=gpu)  # a row stride past F
    _lib.call("iron_gemm_bf16_nt_swiglu", A.data_ptr(), W.data_ptr(), H.data_ptr(), M, F, K, F + 64, s)
    torch.cuda.synchronize()
    assert torch.equal(H[:, :F], ref)
    assert (H[:, F:] == 3.0).all()


@pytest.mark.parametrize("epi", [1, 2, 3, 4, 0x100, 0x102])
def test_skinny_epilogue_matches_tiles(gpu, epi):
    """Activation, clamp and rounding mode as the tiled kernel applies them: on one K step both kernels add the same
    products in one MFMA chain of two links, so only the order inside the 64 products can differ."""
    from iron_amd import _lib

    M, K, N = 16, 64, 256
    A, _, _, W = _inputs(gpu, 64, K, N)
    s = _lib.stream_handle(gpu)
    got, ref = torch.empty(M, N, dtype=BF16, device=gpu), torch.empty(64, N, dtype=BF16, device=gpu)
    for C, m in ((got, M), (ref, 64)):
        _lib.call("iron_gemm_bf16_nt", A.data_ptr(), W.data_ptr(), C.data_ptr(), m, N, K, N, epi, 1, -0.05, 0.2, s)
    torch.cuda.synchronize()
    assert got.float().min() >= -0.0503 and got.float().max() <= 0.2012  # the bounds, one bf16 rounding away
    # two bf16 roundings of sums that differ by a few fp32 ulps: at most two bf16 ulps apart
    d = (got.float() - ref[:M].float()).abs()
    assert (d <= ref[:M].float().abs() * 2.0**-6 + 1e-4).all()


def test_skinny_traced(gpu):
    """A phase trace of the few-row GEMM: one record per workgroup, the output unchanged."""
    from iron_amd import _lib
    from iron_amd.common import tracing_utils as tu

    M, K, N = 13, 512, 200
    A, _, _, W = _inputs(gpu, M, K, N)
    s = _lib.stream_handle(gpu)
    outs = [torch.empty(M, N, dtype=BF16, device=gpu) for _ in range(2)]
    buf = tu.new_buffer(1 << 12, gpu)
    for i, C in enumerate(outs):
        if i:
            tu.arm(buf)
        _lib.call("iron_gemm_bf16_nt", A.data_ptr(), W.data_ptr(), C.data_ptr(), M, N, K, N, 0, 0, 0.0, 0.0, s)
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])
    recs = tu.parse_records(buf)
    assert len(recs) == 13 and all(r["name"] == "gemm_bf16" for r in recs)


# each width of the column tiles, with one and with two stages in flight, ragged
@pytest.mark.parametrize("M,K,N", [(16, 192, 8200), (13, 320, 20488), (9, 128, 28680), (17, 320, 8203), (32, 192, 10240),
                                   (31, 2048, 20488), (20, 2048, 30000), (48, 640, 8192), (40, 64, 4104), (33, 4096, 5001), (9, 2048, 8200)])
def test_skinny_column_tiles(gpu, M, K, N):
    test_skinny_forms(gpu, M, K, N)


@pytest.mark.parametrize("M,K,F", [(16, 128, 8192), (20, 192, 5120), (33, 128, 4096), (48, 320, 4160)])
def test_skinny_pair_stages(gpu, M, K, F):
    test_skinny_swiglu_pair(gpu, M, K, F)


@pytest.mark.parametrize("M,K,N,groups", [
    (4, 128, 4096, 256),  # 16 columns
    (48, 4096, 6144, 192),  # 32: one workgroup per CU, not one and a half of 16
    (16, 512, 20480, 640),
    (32, 2048, 20480, 640),  # a row pitch of whole 4 KiB
    (8, 2112, 16384, 1024),  # 16 again: a long K of few rows
    (13, 2048, 12288, 768),
    (9, 2112, 16384, 256),
    (16, 768, 28672, 448),  # 64
    (31, 2048, 30000, 469),
    (48, 1536, 16384, 256),  # tiles of 64x64 from here on: wide for their rows
    (32, 3072, 16384, 256),
    (32, 192, 30000, 235),  # 128x128
    (32, 1024, 12296, 193),  # 64x64
    (33, 64, 8200, 129),
    (17, 4160, 64, 1),  # a long K
])
def test_skinny_range(gpu, M, K, N, groups):
    """Which kernel takes a call and in how wide columns, by the workgroups of its phase trace: a call goes to the form
    that is faster for it."""
    from iron_amd import _lib
    from iron_amd.common import tracing_utils as tu

    A, _, _, W = _inputs(gpu, M, K, N)
    C, buf = torch.empty(M, N, dtype=BF16, device=gpu), tu.new_buffer(1 << 17, gpu)
    tu.arm(buf)
    _lib.call("iron_gemm_bf16_nt", A.data_ptr(), W.data_ptr(), C.data_ptr(), M, N, K, N, 0, 0, 0.0, 0.0,
              _lib.stream_handle(gpu))
    torch.cuda.synchronize()
    assert len(tu.parse_records(buf)) == groups
    exact = A.double() @ W.double().t()
    bound = exact.abs() * 2.0**-8 + K * 2.0**-23 * (A.double().abs() @ W.double().abs().t())
    assert ((C.double() - exact).abs() <= bound).all()
