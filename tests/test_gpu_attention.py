"""GPU parity of the shared-prefix gated GQA attention and its prep kernel.

Calls the kernels through the operator C ABI (libcujev_ops.so) and compares
with the CPU oracle (oracle/qwen35.py) on the same seeded bf16 inputs.
Tolerance: max |gpu - oracle| / max |oracle| <= 1e-2 on the bf16 outputs
(the target bar for bf16 layer outputs is 2e-2).
"""
import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import qwen35 as orc  # noqa: E402

pytestmark = pytest.mark.gpu
TOL = 1e-2
D = 256


def ops():
    from cujev import ops as o
    o.load()
    return o


def rel_err(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-30))


def bf(x):
    return torch.as_tensor(np.asarray(x, np.float32)).to(torch.bfloat16)


def np32(t):
    return t.float().cpu().numpy()


def make_case(seed, Hq, Hkv, P, seg_lens, stride_tokens=None):
    rng = np.random.default_rng(seed)
    N = int(sum(seg_lens))
    q = orc.bf16_round(rng.standard_normal((N, Hq, D)).astype(np.float32) * 0.6)
    gate = orc.bf16_round(rng.standard_normal((N, Hq, D)).astype(np.float32))
    ks = orc.bf16_round(rng.standard_normal((P, Hkv, D)).astype(np.float32))
    vs = orc.bf16_round(rng.standard_normal((P, Hkv, D)).astype(np.float32))
    ko = orc.bf16_round(rng.standard_normal((N, Hkv, D)).astype(np.float32))
    vo = orc.bf16_round(rng.standard_normal((N, Hkv, D)).astype(np.float32))
    own_base = np.zeros(N, np.int32)
    s = 0
    for L in seg_lens:
        own_base[s: s + L] = s
        s += L
    return q, gate, ks, vs, ko, vo, own_base


def run_attention(o, q, gate, ks, vs, ko, vo, own_base, Hq, Hkv, split=False):
    """split: pass a workspace so that few-workgroup shapes split their key
    tiles over several workgroups and merge the partials."""
    dev = "cuda"
    N, P = q.shape[0], ks.shape[0]
    ps = o.kv_stride(max(P, 1))
    os_ = o.kv_stride(N)
    pk = torch.zeros(Hkv, ps, D, dtype=torch.bfloat16, device=dev)
    pvt = torch.zeros(Hkv, D, ps, dtype=torch.bfloat16, device=dev)
    if P:
        pk[:, :P] = bf(ks.transpose(1, 0, 2)).to(dev)
        pvt[:, :, :P] = bf(vs.transpose(1, 2, 0)).to(dev)
    ok = torch.zeros(Hkv, os_, D, dtype=torch.bfloat16, device=dev)
    ovt = torch.zeros(Hkv, D, os_, dtype=torch.bfloat16, device=dev)
    ok[:, :N] = bf(ko.transpose(1, 0, 2)).to(dev)
    ovt[:, :, :N] = bf(vo.transpose(1, 2, 0)).to(dev)
    # the gate lives in the second half of a fused [q | gate] row per head
    qg = torch.zeros(N, Hq, 2 * D, dtype=torch.bfloat16, device=dev)
    qg[:, :, D:] = bf(gate).to(dev)
    qd = bf(q * orc.LOG2E / 16.0).to(dev)  # the prep kernel's prescaling
    out = torch.empty(N, Hq * D, dtype=torch.bfloat16, device=dev)
    ob = torch.as_tensor(own_base).to(dev)
    ws = None
    if split:
        nb = o.attention_ws_bytes(N, Hq, Hkv, P)
        assert nb > 0, "shape does not split"
        ws = torch.empty(nb, dtype=torch.uint8, device=dev)
    o.attention(qd, qg[:, :, D:], Hq * 2 * D, 2 * D, pk, pvt, P, ps, ok, ovt, os_, ob, Hq, Hkv, out,
                ws=ws)
    torch.cuda.synchronize()
    return np32(out).reshape(N, Hq, D), np32(qd)


def oracle_attention(qd_scaled, gate, ks, vs, ko, vo, own_base):
    # qd_scaled holds bf16(q * log2e / 16); scores in natural-log units are
    # qd.k * ln 2, so the same probabilities as the kernel's exp2.
    return orc.shared_prefix_attention(qd_scaled.astype(np.float64), gate, ks, vs, ko, vo,
                                       own_base, scale=math.log(2.0), bf16_p=True)


CASES = [
    # (seed, Hq, Hkv, P, seg_lens)
    (1, 8, 2, 100, [1, 17, 33]),
    (2, 8, 2, 0, [300]),                  # prefill: P = 0, one causal segment
    (3, 8, 2, 512, [32, 32, 32, 32]),     # config 1 shape (4 branches x 32)
    (4, 16, 4, 64, [16] * 10),            # many short branches, P on a tile edge
    (5, 4, 1, 65, [1] * 40 + [70]),       # one-token branches then a long one
    (6, 8, 2, 1, [5, 64, 2]),
]


@pytest.mark.parametrize("seed,Hq,Hkv,P,seg_lens", CASES)
def test_attention_matches_oracle(seed, Hq, Hkv, P, seg_lens):
    o = ops()
    print(f"case seed={seed} Hq={Hq} Hkv={Hkv} P={P} segs={seg_lens}", flush=True)
    q, gate, ks, vs, ko, vo, ob = make_case(seed, Hq, Hkv, P, seg_lens)
    got, qd = run_attention(o, q, gate, ks, vs, ko, vo, ob, Hq, Hkv)
    ref = oracle_attention(qd, gate, ks, vs, ko, vo, ob)
    err = rel_err(got, ref)
    print(f"rel err {err:.3e}")
    assert err <= TOL


@pytest.mark.parametrize("seed,Hq,Hkv,P,seg_lens", [
    (41, 16, 4, 530, [20, 20, 20, 20]),   # the 4B eval: 12 workgroups -> 9 key splits
    (42, 8, 2, 100, [1, 17, 33]),          # 2 state tiles, own tiles in the last split
    (43, 16, 4, 8192, [1]),                # one token, 16 splits of 8 tiles
    (44, 4, 1, 70, [3, 64, 5]),            # state tile edge; a split of own tiles only
    (45, 16, 4, 0, [200]),                 # a prefill: causal, early rows see few tiles
    (46, 8, 2, 0, [100, 120]),             # two prefill segments
])
def test_attention_key_split_matches_oracle(seed, Hq, Hkv, P, seg_lens):
    """Key tiles split over workgroups with the softmax partials merged: equal
    to the oracle, and to the one-pass kernel up to fp32 summation order."""
    o = ops()
    print(f"key split seed={seed} P={P} seg_lens={seg_lens}", flush=True)
    q, gate, ks, vs, ko, vo, ob = make_case(seed, Hq, Hkv, P, seg_lens)
    got, qd = run_attention(o, q, gate, ks, vs, ko, vo, ob, Hq, Hkv, split=True)
    one, _ = run_attention(o, q, gate, ks, vs, ko, vo, ob, Hq, Hkv)
    ref = oracle_attention(qd, gate, ks, vs, ko, vo, ob)
    e, e1 = rel_err(got, ref), rel_err(got, one)
    print(f"vs oracle {e:.3e}  vs one pass {e1:.3e}")
    assert e <= TOL and e1 <= 1e-2


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("P,seg_lens,pad", [
    (0, [200], {70, 130, 131, 190}),          # amid a causal segment
    (100, [160, 20, 60], {129, 150, 161, 201}),  # and beside segment starts
])
def test_attention_rows_that_see_only_themselves(P, seg_lens, pad, split):
    """own_base[n] = n in rows that are neither the first nor the last of
    their 32: the bases fall again behind them, and each row still sees
    [own_base[n], n] only."""
    o = ops()
    Hq, Hkv = 8, 2
    print(f"padding rows P={P} segs={seg_lens} pad={sorted(pad)} split={split}", flush=True)
    q, gate, ks, vs, ko, vo, ob = make_case(61, Hq, Hkv, P, seg_lens)
    for n in pad:
        ob[n] = n
    got, qd = run_attention(o, q, gate, ks, vs, ko, vo, ob, Hq, Hkv, split=split)
    ref = oracle_attention(qd, gate, ks, vs, ko, vo, ob)
    assert rel_err(got, ref) <= TOL
    for n in pad:
        assert rel_err(got[n], ref[n]) <= TOL, n


@pytest.mark.parametrize("Hq,Hkv,Na,branches", [
    (16, 4, 530, [20] * 4),        # the deferred config-4 pass
    (8, 2, 17, [33, 1, 5]),
    (12, 3, 100, [64, 70]),        # Hkv not dividing 8: plain block mapping
])
def test_attention_pair_equals_two_launches(Hq, Hkv, Na, branches):
    """The paired launch of the deferred-prefill pass: rows [0, Na) are a
    prefill over the state cache's own rows (P = 0), the rest branches over
    those Na keys and their own; the same bits as two one-pass launches."""
    o = ops()
    dev = "cuda"
    rng = np.random.default_rng(Na + len(branches))
    Nb = int(sum(branches))
    N = Na + Nb
    print(f"case Hq={Hq} Hkv={Hkv} Na={Na} branches={branches}", flush=True)
    ps, bs = o.kv_stride(Na), o.kv_stride(Nb)
    pk = torch.zeros(Hkv, ps, D, dtype=torch.bfloat16, device=dev)
    pvt = torch.zeros(Hkv, D, ps, dtype=torch.bfloat16, device=dev)
    pk[:, :Na] = bf(rng.standard_normal((Hkv, Na, D))).to(dev)
    pvt[:, :, :Na] = bf(rng.standard_normal((Hkv, D, Na))).to(dev)
    bk = torch.zeros(Hkv, bs, D, dtype=torch.bfloat16, device=dev)
    bvt = torch.zeros(Hkv, D, bs, dtype=torch.bfloat16, device=dev)
    bk[:, :Nb] = bf(rng.standard_normal((Hkv, Nb, D))).to(dev)
    bvt[:, :, :Nb] = bf(rng.standard_normal((Hkv, D, Nb))).to(dev)
    qd = bf(rng.standard_normal((N, Hq, D)) * 0.6 * orc.LOG2E / 16.0).to(dev)
    qg = torch.zeros(N, Hq, 2 * D, dtype=torch.bfloat16, device=dev)
    qg[:, :, D:] = bf(rng.standard_normal((N, Hq, D))).to(dev)
    base = np.zeros(N, np.int32)
    s0 = 0
    for L in branches:
        base[Na + s0: Na + s0 + L] = s0
        s0 += L
    ob = torch.as_tensor(base).to(dev)
    gate = qg[:, :, D:]
    pair = torch.empty(N, Hq * D, dtype=torch.bfloat16, device=dev)
    o.attention_pair(qd, gate, Hq * 2 * D, 2 * D, pk, pvt, ps, ob, Hq, Hkv, pair, Na, 0, pk, pvt,
                     ps, Na, bk, bvt, bs)
    two = torch.empty_like(pair)
    o.attention(qd[:Na], gate[:Na], Hq * 2 * D, 2 * D, pk, pvt, 0, ps, pk, pvt, ps, ob[:Na], Hq,
                Hkv, two[:Na])
    o.attention(qd[Na:], gate[Na:], Hq * 2 * D, 2 * D, pk, pvt, Na, ps, bk, bvt, bs, ob[Na:], Hq,
                Hkv, two[Na:])
    torch.cuda.synchronize()
    assert torch.isfinite(pair.float()).all()
    assert torch.equal(pair, two)


@pytest.mark.parametrize("Hq,Hkv,Pa,Na,Pb,branches", [
    (16, 4, 0, 530, 300, [20] * 4),        # b sees part of the state: a's rows are the longer
    (8, 2, 700, 40, 64, [33, 1, 5]),       # a over more of the state than b
    (12, 3, 129, 100, 0, [64, 7]),         # Hkv not dividing 8; b without state keys
    (8, 2, 64, 33, 700, [70]),             # b first here
])
def test_attention_pair_in_either_order(Hq, Hkv, Pa, Na, Pb, branches):
    """The paired launch starts the problem with the longer workgroups first.
    Both orders, each problem with state keys and an own-key cache of its own:
    the same bits as two one-pass launches."""
    o = ops()
    dev = "cuda"
    Nb, P = int(sum(branches)), max(Pa, Pb)
    N = Na + Nb
    print(f"pair order Hq={Hq} Pa={Pa} Na={Na} Pb={Pb} branches={branches}", flush=True)
    rng = np.random.default_rng(Na + Pb)
    rnd = lambda *s: bf(rng.standard_normal(s)).to(dev)
    cache = lambda n: (rnd(Hkv, o.kv_stride(n), D), rnd(Hkv, D, o.kv_stride(n)), o.kv_stride(n))
    (pk, pvt, ps), (ak, avt, as_), (bk, bvt, bs) = cache(P), cache(Na), cache(Nb)
    qd = bf(rng.standard_normal((N, Hq, D)) * 0.6 * orc.LOG2E / 16.0).to(dev)
    gate = rnd(N, Hq, D)
    starts = np.cumsum([0] + list(branches[:-1]))
    base = np.concatenate([np.zeros(Na), np.repeat(starts, branches)]).astype(np.int32)
    ob = torch.as_tensor(base).to(dev)
    pair = torch.full((N, Hq * D), float("nan"), dtype=torch.bfloat16, device=dev)
    o.attention_pair(qd, gate, Hq * D, D, pk, pvt, ps, ob, Hq, Hkv, pair, Na, Pa, ak, avt, as_,
                     Pb, bk, bvt, bs)
    two = torch.empty_like(pair)
    o.attention(qd[:Na], gate[:Na], Hq * D, D, pk, pvt, Pa, ps, ak, avt, as_, ob[:Na], Hq, Hkv,
                two[:Na])
    o.attention(qd[Na:], gate[Na:], Hq * D, D, pk, pvt, Pb, ps, bk, bvt, bs, ob[Na:], Hq, Hkv,
                two[Na:])
    torch.cuda.synchronize()
    assert torch.isfinite(pair.float()).all()
    assert torch.equal(pair, two)


def test_attention_branch_isolation():
    """A branch's output does not depend on its siblings. Not bit for bit:
    alone, the branch's rows sit at other positions of the 32-token tiles and
    its own keys start at another offset inside a 64-key tile, which changes
    the order of the fp32 sums (and the split of the state keys), so the
    check is to the kernel's bf16 tolerance."""
    o = ops()
    Hq, Hkv, P = 8, 2, 130
    q, gate, ks, vs, ko, vo, ob = make_case(11, Hq, Hkv, P, [7, 20, 9])
    both, _ = run_attention(o, q, gate, ks, vs, ko, vo, ob, Hq, Hkv)
    # the middle branch alone
    sl = slice(7, 27)
    alone, _ = run_attention(o, q[sl], gate[sl], ks, vs, ko[sl], vo[sl],
                             np.zeros(20, np.int32), Hq, Hkv)
    assert rel_err(alone, both[sl]) <= 1e-2


@pytest.mark.parametrize("seed,q_scale", [(31, 40.0), (32, 120.0)])
def test_attention_scores_beyond_shift_range(seed, q_scale):
    """Scores of tens to hundreds in log2 units, growing along the keys: the
    kernel's softmax shift (0 while the running max stays within 2^+-64)
    moves several times, each move rescaling o and l, and the exponentials
    taken for shift 0 overflow and are redone."""
    o = ops()
    Hq, Hkv, P = 8, 2, 300
    q, gate, ks, vs, ko, vo, ob = make_case(seed, Hq, Hkv, P, [3, 40, 21])
    q = orc.bf16_round(q * (q_scale / 0.6))
    ks = orc.bf16_round(ks * (1.0 + np.arange(P, dtype=np.float32) / 40.0)[:, None, None])
    got, qd = run_attention(o, q, gate, ks, vs, ko, vo, ob, Hq, Hkv)
    smax = float(np.abs(np.einsum("nhd,phd->nhp", qd[:, ::Hq // Hkv], ks)).max())
    print(f"case seed={seed} q_scale={q_scale}: max |score| {smax:.0f} (log2 units)", flush=True)
    assert smax > 4 * 64
    ref = oracle_attention(qd, gate, ks, vs, ko, vo, ob)
    err = rel_err(got, ref)
    print(f"rel err {err:.3e}")
    assert err <= TOL


def test_attention_scores_far_below_zero():
    """Every score near -230 in log2 units: the shift moves down to the first
    tile's max before any key is counted, and every later tile is shifted."""
    o = ops()
    rng = np.random.default_rng(41)
    Hq, Hkv, P, segs = 8, 2, 200, [9, 30]
    N = sum(segs)
    u = rng.standard_normal((Hkv, D)).astype(np.float32)
    ks = orc.bf16_round(u[None] + 0.05 * rng.standard_normal((P, Hkv, D)).astype(np.float32))
    ko = orc.bf16_round(u[None] + 0.05 * rng.standard_normal((N, Hkv, D)).astype(np.float32))
    vs = orc.bf16_round(rng.standard_normal((P, Hkv, D)).astype(np.float32))
    vo = orc.bf16_round(rng.standard_normal((N, Hkv, D)).astype(np.float32))
    gate = orc.bf16_round(rng.standard_normal((N, Hq, D)).astype(np.float32))
    heads = np.arange(Hq) // (Hq // Hkv)
    q = orc.bf16_round(-10.0 * u[heads][None] +
                       0.05 * rng.standard_normal((N, Hq, D)).astype(np.float32))
    ob = np.concatenate([np.full(L, s, np.int32) for s, L in zip(np.cumsum([0] + segs[:-1]), segs)])
    got, qd = run_attention(o, q, gate, ks, vs, ko, vo, ob, Hq, Hkv)
    smax = float(np.einsum("nhd,phd->nhp", qd[:, ::Hq // Hkv], ks).max())
    print(f"largest score {smax:.0f} (log2 units)", flush=True)
    assert smax < -2 * 64
    ref = oracle_attention(qd, gate, ks, vs, ko, vo, ob)
    err = rel_err(got, ref)
    print(f"rel err {err:.3e}")
    assert err <= TOL


def test_attn_prep_matches_oracle():
    o = ops()
    rng = np.random.default_rng(21)
    Hq, Hkv, N, rot, theta, eps = 8, 2, 150, 64, 1e7, 1e-6  # positions up to 8000 below
    W = Hq * 2 * D + 2 * Hkv * D
    proj = orc.bf16_round(rng.standard_normal((N, W)).astype(np.float32))
    qn = (1.0 + 0.1 * rng.standard_normal(D)).astype(np.float32)
    kn = (1.0 + 0.1 * rng.standard_normal(D)).astype(np.float32)
    pos = (np.arange(N) * 53 + 11).astype(np.int32)
    stride = o.kv_stride(N)
    dev = "cuda"
    qs = orc.LOG2E / 16.0
    q_out = torch.empty(N, Hq, D, dtype=torch.bfloat16, device=dev)
    kc = torch.zeros(Hkv, stride, D, dtype=torch.bfloat16, device=dev)
    vtc = torch.zeros(Hkv, D, stride, dtype=torch.bfloat16, device=dev)
    rope = o.rope_table(theta, rot, int(pos.max()) + 1)
    o.attn_prep(bf(proj).to(dev), torch.as_tensor(qn).to(dev), torch.as_tensor(kn).to(dev),
                torch.as_tensor(pos).to(dev), Hq, Hkv, rot, rope, eps, qs, q_out, kc, vtc, stride)
    torch.cuda.synchronize()
    rq, rg, rk, rv = orc.attn_prep(proj, qn, kn, pos, Hq, Hkv, rot, theta, eps)
    assert rel_err(np32(q_out), rq * qs) <= 1e-2
    assert rel_err(np32(kc)[:, :N].transpose(1, 0, 2), rk) <= 1e-2
    # V is copied bit-exactly, transposed
    np.testing.assert_array_equal(np32(vtc)[:, :, :N].transpose(2, 0, 1), rv.astype(np.float32))


@pytest.mark.parametrize("Na,Nb", [(530, 80), (17, 33), (4, 1)])
def test_attn_prep_pair_equals_two_launches(Na, Nb):
    """The deferred-prefill pass's prep: rows [0, Na) into the state cache,
    the rest into the branch scratch at their own columns; the same bits as
    two launches (Na not a multiple of the 4-token workgroup included)."""
    o = ops()
    rng = np.random.default_rng(Na * 3 + Nb)
    Hq, Hkv, rot, theta, eps = 16, 4, 64, 1e7, 1e-6
    N = Na + Nb
    W = Hq * 2 * D + 2 * Hkv * D
    dev = "cuda"
    proj = bf(rng.standard_normal((N, W))).to(dev)
    qn = torch.as_tensor((1.0 + 0.1 * rng.standard_normal(D)).astype(np.float32)).to(dev)
    kn = torch.as_tensor((1.0 + 0.1 * rng.standard_normal(D)).astype(np.float32)).to(dev)
    pos = torch.as_tensor(np.concatenate([np.arange(Na), Na + np.arange(Nb) % 7]).astype(np.int32)).to(dev)
    rope = o.rope_table(theta, rot, N + 8)
    qs = orc.LOG2E / 16.0
    sa, sb = o.kv_stride(Na), o.kv_stride(Nb)

    def bufs():
        return (torch.empty(N, Hq, D, dtype=torch.bfloat16, device=dev),
                torch.zeros(Hkv, sa, D, dtype=torch.bfloat16, device=dev),
                torch.zeros(Hkv, D, sa, dtype=torch.bfloat16, device=dev),
                torch.zeros(Hkv, sb, D, dtype=torch.bfloat16, device=dev),
                torch.zeros(Hkv, D, sb, dtype=torch.bfloat16, device=dev))
    q1, ka, va, kb, vb = bufs()
    o.attn_prep_pair(proj, qn, kn, pos, Na, Hq, Hkv, rot, rope, eps, qs, q1, ka, va, sa, kb, vb, sb)
    q2, ka2, va2, kb2, vb2 = bufs()
    o.attn_prep(proj[:Na], qn, kn, pos[:Na], Hq, Hkv, rot, rope, eps, qs, q2[:Na], ka2, va2, sa)
    o.attn_prep(proj[Na:], qn, kn, pos[Na:], Hq, Hkv, rot, rope, eps, qs, q2[Na:], kb2, vb2, sb)
    torch.cuda.synchronize()
    for x, y in ((q1, q2), (ka, ka2), (va, va2), (kb, kb2), (vb, vb2)):
        assert torch.equal(x, y)


@pytest.mark.parametrize("rows", [64])
def test_attention_capacity_shape(rows):
    """Config 3 shape (Hq 16 / Hkv 4, state 8192, 256 branches x 16) against a
    torch fp32 reference on the device, plus the CPU oracle on a row sample."""
    o = ops()
    Hq, Hkv, P = 16, 4, 8192
    segs = [16] * 256
    N = sum(segs)
    g = torch.Generator(device="cpu").manual_seed(1)
    dev = "cuda"
    ps, os_ = o.kv_stride(P), o.kv_stride(N)
    pk = torch.zeros(Hkv, ps, D, dtype=torch.bfloat16, device=dev)
    pvt = torch.zeros(Hkv, D, ps, dtype=torch.bfloat16, device=dev)
    ok = torch.zeros(Hkv, os_, D, dtype=torch.bfloat16, device=dev)
    ovt = torch.zeros(Hkv, D, os_, dtype=torch.bfloat16, device=dev)
    ks = torch.randn(Hkv, P, D, generator=g).to(torch.bfloat16)
    vs = torch.randn(Hkv, P, D, generator=g).to(torch.bfloat16)
    ko = torch.randn(Hkv, N, D, generator=g).to(torch.bfloat16)
    vo = torch.randn(Hkv, N, D, generator=g).to(torch.bfloat16)
    qd = (torch.randn(N, Hq, D, generator=g) * (orc.LOG2E / 16.0)).to(torch.bfloat16)
    gate = torch.randn(N, Hq, D, generator=g).to(torch.bfloat16)
    pk[:, :P] = ks.to(dev)
    pvt[:, :, :P] = vs.transpose(1, 2).to(dev)
    ok[:, :N] = ko.to(dev)
    ovt[:, :, :N] = vo.transpose(1, 2).to(dev)
    ob = torch.as_tensor(np.repeat(np.arange(0, N, 16), 16).astype(np.int32)).to(dev)
    out = torch.empty(N, Hq * D, dtype=torch.bfloat16, device=dev)
    gd = gate.to(dev)
    o.attention(qd.to(dev), gd, Hq * D, D, pk, pvt, P, ps, ok, ovt, os_, ob, Hq, Hkv, out)
    torch.cuda.synchronize()
    got = out.float().view(N, Hq, D)
    # torch fp32 reference on the device, per kv-head, chunked over tokens
    ref = torch.empty(N, Hq, D, device=dev)
    kst, vst = ks.float().to(dev), vs.float().to(dev)
    kof, vof = ko.float().to(dev), vo.float().to(dev)
    qf = qd.float().to(dev) * math.log(2.0)
    own_mask = torch.full((16, 16), float("-inf"), device=dev).triu(1)
    for kh in range(Hkv):
        for b in range(256):
            sl = slice(16 * b, 16 * b + 16)
            kk = torch.cat([kst[kh], kof[kh, sl]], 0)
            vv = torch.cat([vst[kh], vof[kh, sl]], 0)
            qq = qf[sl, 4 * kh: 4 * kh + 4]  # [16, 4, D]
            s = torch.einsum("thd,kd->htk", qq, kk)
            s[:, :, P:] += own_mask
            p = torch.softmax(s, -1)
            ref[sl, 4 * kh: 4 * kh + 4] = torch.einsum("htk,kd->thd", p, vv)
    ref = ref * torch.sigmoid(gd.float())
    err = float((got - ref).abs().max() / ref.abs().max())
    print(f"capacity rel err vs torch fp32: {err:.3e}")
    assert err <= TOL
    # oracle on a sample of rows
    rng = np.random.default_rng(0)
    rows_idx = np.sort(rng.choice(N, rows, replace=False))
    ksn, vsn = np32(ks).transpose(1, 0, 2), np32(vs).transpose(1, 0, 2)
    kon, von = np32(ko).transpose(1, 0, 2), np32(vo).transpose(1, 0, 2)
    qn, gn, obn = np32(qd), np32(gate), ob.cpu().numpy()
    worst = 0.0
    for n in rows_idx:
        b = int(obn[n])
        # the branch's tokens b..n, own keys b..n; keep the last row
        r = orc.shared_prefix_attention(qn[b:n + 1].astype(np.float64), gn[b:n + 1], ksn, vsn,
                                        kon[b:n + 1], von[b:n + 1],
                                        np.zeros(n + 1 - b, np.int32),
                                        scale=math.log(2.0), bf16_p=True)[-1:]
        worst = max(worst, rel_err(got[n:n + 1].cpu().numpy(), r))
    print(f"capacity rel err vs oracle sample: {worst:.3e}")
    assert worst <= TOL
