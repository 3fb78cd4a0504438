"""The reference-shaped call's rows as cut on the device, into equal parts of a
smallest length that depends on the rows and the cache type (resolve() in
attention_decode_wg.h), against the oracle: partition edges, one row, rows of
one sequence, more rows than a workgroup has threads, and rows whose equal parts
exceed the smallest partition. Two-term weights: split rows of a 16-bit cache
are as exact as the query's rounding lets them be."""
import numpy as np
import pytest
import torch

from cases import make_case
from gpu_util import oracle_out, poison_unused
from test_gpu_attention import run_decode, tol_for, within

pytestmark = pytest.mark.gpu

EDGES = [1, 255, 256, 257, 511, 512, 513, 1024, 1025, 40]  # a partition's 256, 512 or 1024 keys at least


@pytest.mark.parametrize("heads,kv,bs", [((14, 2, 64), "f32", 16), ((14, 2, 64), "bf16", 8), ((32, 8, 128), "f16", 16),
                                         ((16, 16, 64), "bf16", 64), ((8, 8, 128), "f32", 16)])
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


@pytest.mark.parametrize("heads,kv", [((32, 8, 128), "f16"), ((14, 2, 64), "bf16"), ((8, 8, 128), "bf16")])
def test_unplanned_weights_are_not_rounded(gpu, heads, kv):
    """Queries that the cache type holds exactly: what is left of the error is the weights' second term (2^-17 of them
    in bf16, 2^-23 in fp16) and fp32 sums, far below one rounding of the weights (2^-9 and 2^-12)."""
    H, KH, hd = heads
    case = make_case([3000, 100, 1500, 2200, 700, 900], H, KH, hd, 16, seed=6, kv_bf16=kv == "bf16", kv_f16=kv == "f16")
    q = torch.from_numpy(case.q).to(torch.bfloat16 if kv == "bf16" else torch.float16)
    case.q = q.float().numpy()
    got, qh = run_decode(case, torch.float32, gpu)
    want = oracle_out(case, qh)
    rel = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"{heads} {kv}: relative error {rel:.2e}")
    assert rel < (2.0 ** -15 if kv == "bf16" else 2.0 ** -19)
