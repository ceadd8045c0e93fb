"""GPU parity of the 256-row tiles of cujev_op_gemm_wide (gemm_block.hip: both
operands staged by DMA): bit for bit against tile (4, 10), which keeps its own
kernel and walks K in the same order, at the edges of the tiles (one token, one
past a tile, rows past M, one K chunk, several rounds of workgroups), and
against float32 references (1e-2 of the largest value: the bf16 output
rounding, 2^-9, and fp32 summation order)."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def ops():
    from cujev import ops as o
    o.load()
    return o


def rand_bf16(*shape, seed, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(*shape, device="cuda", generator=g) * scale).to(torch.bfloat16)


@pytest.mark.parametrize("N,M,K", [(1, 256, 128), (129, 272, 256), (193, 2608, 384),
                                   (257, 512, 1152), (1031, 18432, 256), (4500, 4112, 128)])
@pytest.mark.parametrize("ng", [8, 12, 16])
def test_block_tiles_equal_the_wide_tile(N, M, K, ng):
    o = ops()
    X, W = rand_bf16(N, K, seed=21), rand_bf16(M, K, seed=22, scale=0.05)
    Wt = o.gemm_small_tile(W)
    ref = torch.empty(N, M, dtype=torch.bfloat16, device="cuda")
    o.gemm_wide(X, Wt, Y=ref, rg=4, ng=10)
    Yb = torch.full((N, M + 24), 7.0, dtype=torch.bfloat16, device="cuda")
    o.gemm_wide(X, Wt, Y=Yb[:, :M], rg=4, ng=ng)
    torch.cuda.synchronize()
    assert torch.equal(Yb[:, :M], ref)
    assert (Yb[:, M:] == 7.0).all()  # nothing past the row's M outputs
    f = X.float() @ W.float().t()
    assert float((ref.float() - f).abs().max() / f.abs().max()) <= 1e-2


@pytest.mark.parametrize("N,I,K", [(1, 160, 128), (130, 144, 256), (257, 9216, 256)])
@pytest.mark.parametrize("ng", [12, 16])
def test_block_tiles_gated(N, I, K, ng):
    o = ops()
    X, W = rand_bf16(N, K, seed=23), rand_bf16(2 * I, K, seed=24, scale=0.05)
    Wt = o.gemm_small_tile(W)
    ref = torch.empty(N, I, dtype=torch.bfloat16, device="cuda")
    act = torch.full((N, I), float("nan"), dtype=torch.bfloat16, device="cuda")
    o.gemm_wide(X, Wt, Y=ref, gated=True, rg=4, ng=10)
    o.gemm_wide(X, Wt, Y=act, gated=True, rg=4, ng=ng)
    torch.cuda.synchronize()
    assert torch.equal(act, ref)


@pytest.mark.parametrize("N,M,K,splits", [(1, 256, 256, 2), (300, 528, 768, 3), (611, 2560, 1024, 8)])
@pytest.mark.parametrize("ng", [8, 12, 16])
def test_block_tiles_partials(N, M, K, splits, ng):
    o = ops()
    X, Wt = rand_bf16(N, K, seed=25), o.gemm_small_tile(rand_bf16(M, K, seed=26, scale=0.05))
    ref = torch.empty(splits, N, M, device="cuda")
    P = torch.full((splits, N, M), float("nan"), device="cuda")
    o.gemm_wide(X, Wt, P=ref, splits=splits, rg=4, ng=10)
    o.gemm_wide(X, Wt, P=P, splits=splits, rg=4, ng=ng)
    torch.cuda.synchronize()
    assert torch.equal(P, ref)


@pytest.mark.parametrize("shift,ldx,ldy", [(0, 388, 272), (4, 392, 272), (0, 384, 276),
                                           (0, 384, 273)])
def test_block_tiles_take_rows_of_any_alignment(shift, ldx, ldy):
    """X rows that are not whole 16-byte pieces run another tile, output rows
    that are not leave by 2-byte stores: the same bits."""
    o = ops()
    N, M, K = 70, 272, 384
    X = rand_bf16(N, ldx + shift, seed=27)[:, shift:shift + K]
    W = rand_bf16(M, K, seed=28, scale=0.05)
    Wt = o.gemm_small_tile(W)
    ref = torch.empty(N, M, dtype=torch.bfloat16, device="cuda")
    o.gemm_wide(X.contiguous(), Wt, Y=ref, rg=4, ng=10)
    for ng in (8, 12, 16):
        Y = torch.empty(N, ldy, dtype=torch.bfloat16, device="cuda")[:, :M]
        o.gemm_wide(X, Wt, Y=Y, rg=4, ng=ng)
        torch.cuda.synchronize()
        assert torch.equal(Y, ref), ng
