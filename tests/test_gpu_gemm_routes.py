"""Which kernels run an engine's projections past 96 tokens, seen from the
hipBLASLt plans that a process prints as it makes them (CUJEV_GEMM_DEBUG): the
tiled kernels by default, hipBLASLt where its table was tuned for exactly the
call's tokens, and hipBLASLt for all of them with CUJEV_WIDE_GEMM=0. Results
on every route within the engine tests' 3e-3 in probability of the default's,
and every repeat of an eval (eager, captured, replayed) the same bits.

The switches are read once per process, so each route has a process of its own.
"""
import os
import re
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from cujev import gemm_tune, ops, synthetic  # noqa: E402

pytestmark = pytest.mark.gpu
PROB_TOL = 3e-3
PKG = Path(ops.__file__).resolve().parents[1]
BRANCHES, LEN = 33, 65
N = BRANCHES * LEN  # 2145 tokens: past the limit below which the tiled kernels always run

CHILD = """
import sys
import numpy as np
import torch  # the hipBLASLt whose version the table names
from cujev import Branch, Engine
ckpt, out, B, L = sys.argv[1], sys.argv[2], int(sys.argv[3]), int(sys.argv[4])
rng = np.random.default_rng(5)
ids = lambda n: [int(x) for x in rng.integers(16, 4096, size=n)]
e = Engine(ckpt, max_state_tokens=256, max_branch_tokens=B * L, max_branches=64, max_candidates=8)
e.prefill(ids(200))
br = [Branch(ids(L), ids(8)) for _ in range(B)]
np.save(out, np.array([e.eval(br) for _ in range(5)]))
e.close()
"""


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    d = tmp_path_factory.mktemp("routes")
    # the tiny preset with the large models' GDN heads (an in_proj of a multiple
    # of 64 rows is tiled too), a down projection of a shape of its own, and a layer
    # behind the attention layer (the last one runs on the branches' last rows)
    cfg = synthetic.make_config(**dict(synthetic.PRESETS["tiny"], lin_k_heads=16, lin_v_heads=32,
                                       intermediate_size=1152, num_layers=5))
    synthetic.write_checkpoint(d / "ckpt", cfg, seed=0, norm_std=0.1)
    return d, cfg


def run(model, name, **kw):
    """(logits of 5 repeats, {(N, M, K): how hipBLASLt was planned})"""
    d, _ = model
    print(f"route {name}", flush=True)
    e = dict(os.environ, PYTHONPATH=str(PKG), CUJEV_GEMM_DEBUG="1", **kw)
    out = d / f"{name}.npy"
    r = subprocess.run([sys.executable, "-c", CHILD, str(d / "ckpt"), str(out), str(BRANCHES),
                        str(LEN)], env=e, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    plans = {tuple(map(int, m[:3])): m[3] for m in
             re.findall(r"gemm plan N=(\d+) M=(\d+) K=(\d+) f32out=0: (.*)", r.stderr)}
    x = np.load(out)
    for i in range(1, len(x)):
        np.testing.assert_array_equal(x[i], x[0])
    return x[0].astype(np.float64), plans


def probabilities(x):
    p = np.exp(x - x.max(-1, keepdims=True))
    return p / p.sum(-1, keepdims=True)


@pytest.fixture(scope="module")
def default(model):
    return run(model, "default", CUJEV_GEMM_TABLE="/nonexistent")


def projections(cfg):
    return {(M, K) for M, K in gemm_tune.projection_shapes(cfg)}


def test_tiled_kernels_run_without_an_entry(model, default):
    cfg = model[1]
    assert not {(m, k) for n, m, k in default[1] if n > 96} & projections(cfg)


def test_an_entry_for_the_calls_tokens_goes_to_hipblaslt(model, default):
    """qkv, gate|up and out_proj are tuned for N, in_proj for N + 32 only. The
    first runs on hipBLASLt, and gate|up, whose plan is not a 256-row tile of 192
    tokens or more; not out_proj (its plan splits K), nor in_proj (a
    neighbour's entry)."""
    d, cfg = model
    ops.load()
    (qkv, H), _, (inp, _), (_, vd), (gu, _), _ = gemm_tune.projection_shapes(cfg)
    assert ops.gemm_plan(N, qkv, H)[2] == 1 and ops.gemm_plan(N, inp, H)[2] == 1
    assert ops.gemm_plan(N, gu, H, True)[:2] not in {(4, 12), (4, 16)}
    assert ops.gemm_plan(N, H, vd, False, 8)[2] > 1
    W = torch.randn(qkv, H, device="cuda").to(torch.bfloat16)
    X = torch.randn(N, H, device="cuda").to(torch.bfloat16)
    idx, _, _ = ops.gemm_tune(X, W, torch.empty(N, qkv, device="cuda", dtype=torch.bfloat16))
    table = d / "table.txt"
    table.write_text(f"# hipblaslt {ops.blaslt_version()}\n{N} {qkv} {H} 0 {idx}\n"
                     f"{N + 32} {inp} {H} 0 {idx}\n{N} {gu} {H} 0 {idx}\n{N} {H} {vd} 0 {idx}\n")
    x, plans = run(model, "tuned", CUJEV_GEMM_TABLE=str(table))
    big = {k for k in plans if k[0] > 96 and k[1:] in projections(cfg)}
    assert big == {(N, qkv, H), (N, gu, H)} and plans[(N, qkv, H)] == "tuned table"
    assert np.abs(probabilities(x) - probabilities(default[0])).max() <= PROB_TOL


def test_wide_gemm_off_runs_every_projection_on_hipblaslt(model, default):
    """The fallback of shapes that the tiled copy does not cover: plain
    projections, the residual ones and the unfused gate|up + silu_mul, in the
    prefill of 200 tokens and the eval of 2145."""
    cfg = model[1]
    x, plans = run(model, "library", CUJEV_GEMM_TABLE="/nonexistent", CUJEV_WIDE_GEMM="0")
    for n in (200, N):
        assert {(m, k) for m_n, m, k in plans if m_n == n} >= projections(cfg)
    assert np.abs(probabilities(x) - probabilities(default[0])).max() <= PROB_TOL
