"""The reference-shaped call's rows as cut on the device from the step's
positions (resolve() in attention_decode_wg.h), against the oracle: partition
edges, one row, rows of one sequence, more rows than a workgroup has threads,
and a step whose share of keys exceeds the smallest partition."""
import numpy as np
import pytest
import torch

from cases import make_case
from gpu_util import oracle_out, poison_unused
from test_gpu_attention import run_decode, tol_for, within

pytestmark = pytest.mark.gpu

EDGES = [1, 255, 256, 257, 511, 512, 513, 1024, 1025, 40]  # 256 keys (fp32) and 512 a partition at least


@pytest.mark.parametrize("heads,kv,bs", [((14, 2, 64), "f32", 16), ((14, 2, 64), "bf16", 8), ((32, 8, 128), "f16", 16),
                                         ((16, 16, 64), "bf16", 64)])
@pytest.mark.parametrize("kind", ["edges", "one", "chunk", "many", "share"])
def test_unplanned_rows(gpu, heads, kv, bs, kind):
    H, KH, hd = heads
    rng = np.random.default_rng(H)
    ctx = {"edges": EDGES, "one": [2300], "chunk": [700, 90], "many": list(rng.integers(1, 90, 259)) + [1500],
           "share": [9000, 4100, 8000, 30] * (1 if KH > 8 else 2)}[kind]
    q_len = [60, 3] if kind == "chunk" else None
    case = make_case(ctx, H, KH, hd, bs, q_len=q_len, seed=len(ctx), kv_bf16=kv == "bf16", kv_f16=kv == "f16")
    poison_unused(case)
    got, qh = run_decode(case, torch.float32, gpu)
    want = oracle_out(case, qh)
    assert np.isfinite(got).all() and within(got, want, tol_for(case, qh, want))
