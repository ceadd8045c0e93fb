"""GPU parity of the one-launch form of the GDN scan (evals whose segments are
one chunk each and write no state back) against the general two-launch path on
the same inputs.

Both take the same fragments, split products and order of operations, so the
outputs are equal bit for bit: the tolerance is zero. Sizes: the edges of the
16-row and 32-row tiles, one, two, three and four v-heads per k-head (a pair
with and without its second v-head), unit counts that are and are not a
multiple of 8 (the workgroup order differs), with and without a state and a
conv tail, z rows and a state that are not 16-byte aligned.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from test_gpu_gdn import DK, DV, Layer, bf, ops, run_gpu  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("seg_lens,Hk,Hv,state", [
    ([1, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64], 2, 4, True),
    ([64, 1, 3, 33], 4, 12, True),
    ([5, 16, 64], 4, 4, True),
    ([16] * 9, 8, 16, True),
    ([2, 40], 4, 16, True),
    ([7, 64, 30], 8, 8, False)])
def test_one_launch_equals_general_path(seg_lens, Hk, Hv, state, fused):
    o = ops()
    print(f"one chunk seg_lens={seg_lens} Hk={Hk} Hv={Hv} state={state} fused={fused}", flush=True)
    L = Layer(41, Hk, Hv)
    br = L.proj(sum(seg_lens))
    kw = {}
    if state:
        kw = {"conv_in": L.rng.standard_normal((L.C, 3)).astype(np.float32),
              "S_in": L.rng.standard_normal((Hv, DK, DV)).astype(np.float32)}
    got = run_gpu(o, L, br, seg_lens, fused=fused, **kw)
    ref = run_gpu(o, L, br, seg_lens, fused=fused, tell_max=False, **kw)
    assert np.isfinite(ref["y"]).all()
    np.testing.assert_array_equal(got["y"], ref["y"])


@pytest.mark.parametrize("off,s_off", [(0, 0), (1, 1), (4, 2)])
def test_one_launch_unaligned_operands(off, s_off):
    """z rows `off` elements into rows of a stride that is no multiple of 8,
    the state s_off floats into its buffer."""
    o = ops()
    print(f"one chunk, z offset {off}, state offset {s_off}", flush=True)
    seg_lens, Hk, Hv = [33, 20, 64], 2, 4
    L, N, dev = Layer(43, Hk, Hv), sum(seg_lens), "cuda"
    rng = L.rng
    t = lambda a: torch.as_tensor(a).to(dev)
    q, k = (t(rng.standard_normal((N, Hk, DK)).astype(np.float32) / 11) for _ in range(2))
    v = t(rng.standard_normal((N, Hv, DV)).astype(np.float32))
    g = t(-np.abs(rng.standard_normal((N, Hv))).astype(np.float32))
    beta = t(rng.uniform(0, 1, (N, Hv)).astype(np.float32))
    z = torch.zeros(N, Hv * DV + off, dtype=torch.bfloat16, device=dev)
    z[:, off:] = bf(rng.standard_normal((N, Hv * DV))).to(dev)
    sbuf = torch.zeros(Hv * DK * DV + 4, dtype=torch.float32, device=dev)
    S = sbuf[s_off: s_off + Hv * DK * DV]
    S.copy_(t(rng.standard_normal(Hv * DK * DV).astype(np.float32)))
    tok0, clen, seg0, segn = (t(a) for a in o.chunk_table(seg_lens))
    scratch = torch.empty(o.gdn_scratch_bytes(len(seg_lens), Hv, N), dtype=torch.uint8, device=dev)
    res = []
    for msc in (1, 0):
        y = torch.full((N, Hv * DV), float("nan"), dtype=torch.bfloat16, device=dev)
        o.gdn_scan(q, k, v, g, beta, tok0, clen, seg0, segn, S, None, z[:, off:], z.stride(0),
                   t(L.norm_w), L.eps, Hk, Hv, y, scratch, max_seg_chunks=msc)
        torch.cuda.synchronize()
        res.append(y.float().cpu().numpy())
    assert np.isfinite(res[1]).all()
    np.testing.assert_array_equal(res[0], res[1])


@pytest.mark.parametrize("packed", [False, True])
def test_one_launch_chunks_without_tokens(packed):
    """Chunks of length 0 (a table of a fixed size, a branch without tokens)
    before, between and behind the others: nothing is read or written for
    them, the other rows are the same bits."""
    o = ops()
    print(f"one chunk, empty chunks, packed={packed}", flush=True)
    Hk, Hv, N, dev = 2, 4, 53, "cuda"
    L = Layer(47, Hk, Hv)
    pd = bf(L.proj(N)).to(dev)
    t = lambda a, dt: torch.as_tensor(np.asarray(a, dt)).to(dev)
    f = lambda a: t(a, np.float32)
    base = t(np.repeat([0, 33], [33, 20]), np.int32)
    cin, S = f(L.rng.standard_normal((L.C, 3))), f(L.rng.standard_normal((Hv, DK, DV)))
    res = []
    for tok0, clen in (([0, 33], [33, 20]), ([0, 0, 33, 33, 53], [0, 33, 0, 20, 0])):
        n = len(tok0)
        y = torch.full((N, Hv * DV), float("nan"), dtype=torch.bfloat16, device=dev)
        scratch = torch.empty(o.gdn_scratch_bytes(n, Hv, N), dtype=torch.uint8, device=dev)
        o.gdn_layer(pd, f(L.conv_w), cin, None, 0, base, f(L.A_neg), f(L.dt_bias),
                    t(tok0, np.int32), t(clen, np.int32),
                    None if packed else t(range(n), np.int32),
                    None if packed else t([1] * n, np.int32), S, None, f(L.norm_w), L.eps, Hk, Hv,
                    y, scratch, max_seg_chunks=1,
                    chunk_starts=t([1] * n, np.int64) if packed else None)
        torch.cuda.synchronize()
        res.append(y.float().cpu().numpy())
    assert np.isfinite(res[0]).all()
    np.testing.assert_array_equal(res[1], res[0])
