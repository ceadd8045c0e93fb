"""Attention shapes past the smallest evals whose leftover workgroups share
out their key tiles (cujev_op_attention_ws): against the one-pass kernel. P
is rounded to bf16 at the same points in both (the softmax shift stays 0), so
they differ by fp32 summation order and one bf16 rounding of the output:
at most 2^-8 of the largest value."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
D = 256


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv,P,lens", [
    (16, 4, 1500, [40] * 16),           # 80 workgroups, all shared
    (16, 4, 2048, [33] * 64 + [1]),     # 8 workgroups past a whole round
    (16, 4, 1100, [64] * 34),           # 16 past it, branches of two tiles
    (12, 3, 1300, [50] * 8),            # Hkv not dividing 8, all shared
    (12, 3, 1984, [128] * 22),          # and 264 workgroups: 9 past 85 whole tiles
    (4, 1, 900, [7] * 100),             # one kv-head over the 8 XCDs
    (16, 4, 1160, [4] * 163 + [2]),     # 21 tiles: 3 shares each would crowd an XCD
    (16, 4, 700, [32] * 5),             # as would 12 of 5 tiles, in the smallest evals' rule
])
def test_shared_key_tiles_equal_one_pass(Hq, Hkv, P, lens):
    compare(Hq, Hkv, P, lens)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 7, 8, 9, 16, 17, 24, 25, 31, 32, 33])
def test_partials_of_tiles_of_any_length(n):
    """Partials leave row by row from another row in each wave: every row of a
    tile of n tokens is written (the workspace is NaN until then)."""
    compare(8, 2, 700, [n])


def compare(Hq, Hkv, P, lens):
    from cujev import ops
    ops.load()
    N = sum(lens)
    print(f"shares Hq={Hq} Hkv={Hkv} P={P} N={N}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(N)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).to(torch.bfloat16)
    ps, os_ = ops.kv_stride(P), ops.kv_stride(N)
    q = (torch.randn(N, Hq, D, device="cuda", generator=g) * 0.09).to(torch.bfloat16)
    gate, pk, pvt = rnd(N, Hq, D), rnd(Hkv, ps, D), rnd(Hkv, D, ps)
    ok, ovt = rnd(Hkv, os_, D), rnd(Hkv, D, os_)
    starts = np.concatenate([[0], np.cumsum(lens)[:-1]])
    own = torch.as_tensor(np.repeat(starts, lens).astype(np.int32)).cuda()
    outs = []
    nb = ops.attention_ws_bytes(N, Hq, Hkv, P)
    assert nb > 0, "shape does not split"
    ws = torch.full((nb,), 0xFF, dtype=torch.uint8, device="cuda")  # NaN until written
    for w in (None, ws):
        out = torch.full((N, Hq * D), float("nan"), dtype=torch.bfloat16, device="cuda")
        ops.attention(q, gate, Hq * D, D, pk, pvt, P, ps, ok, ovt, os_, own, Hq, Hkv, out, ws=w)
        torch.cuda.synchronize()
        outs.append(out.float())
    assert torch.isfinite(outs[1]).all()
    assert float((outs[0] - outs[1]).abs().max()) <= 2 ** -8 * float(outs[0].abs().max())



def test_partials_fit_the_static_scratch():
    """Every shape's partials fit the no-allocation entry point's array, and
    shapes of whole rounds of workgroups do not split."""
    from cujev import ops
    for Hkv in (1, 2, 3, 4, 8):
        for P in (0, 1, 64, 530, 1024, 8192, 100000):
            for N in [*range(1, 300), *range(300, 12289, 97), 2048, 4096, 8192]:
                assert ops.attention_ws_bytes(N, 4 * Hkv, Hkv, P) <= 33816576
    assert ops.attention_ws_bytes(2048, 16, 4, 8192) == 0
    assert ops.attention_ws_bytes(4096, 16, 4, 8192) == 0
    assert ops.attention_ws_bytes(2560, 16, 4, 8192) > 0
