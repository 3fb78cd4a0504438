"""GPU parity of the prefill tiles (attention_prefill_wg.h, and
attention_prefill_f32_wg.h for fp32 caches) with the oracle at
the edges of their tiles, partitions and softmax base."""
import numpy as np
import pytest
import torch

import oracle
from cases import make_case
from gpu_util import emulated_bar, max_abs, oracle_out, poison_unused
from llm_engine_amd._lib import LE_PLAN_XCD_LOCAL
from test_gpu_attention import TOL_F32, run_ragged, within

pytestmark = pytest.mark.gpu

# 16-bit activations round the output once more (2^-9 and 2^-12 relative,
# doubled for the error carried into it)
OUT_REL = {"f32": 0.0, "bf16": 2.0 ** -8, "f16": 2.0 ** -11}
ACT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def check(case, act, gpu, want_split=None, want_wide=False, bar=None, flags=LE_PLAN_XCD_LOCAL):
    got, qh, plan = run_ragged(case, ACT[act], gpu, flags=flags)
    assert plan.plan.cfg.chunk_q_tile == (-1 if want_wide else 0)
    if want_split is not None:
        assert (plan.plan.n_parts > 0) == want_split
    want = oracle_out(case, qh)
    tol = emulated_bar(case, qh, want) if bar is None else bar(qh, want)
    err = np.abs(got.astype(np.float64) - want)
    print(f"prefill {case.q_heads}/{case.kv_heads}x{case.head_dim} bs {case.block_size} rows {case.n_tokens} "
          f"items {plan.plan.n_chunk_items} parts {plan.plan.n_parts}: max|err| {err.max():.3e} tol {tol:.3e}")
    assert np.isfinite(got).all() and (err <= tol + OUT_REL[act] * np.abs(want)).all()
    return got


# rows of a 128-column tile: 18 (G 7), 16 (G 8), 128 (G 1), 32 (G 4); keys at
# the edges of the 64-key tiles, of a block and of the causal diagonal
@pytest.mark.parametrize("heads,kv,act,bs", [((14, 2, 64), "bf16", "bf16", 16), ((32, 4, 64), "f16", "f16", 8),
                                             ((3, 3, 64), "bf16", "f32", 32), ((32, 8, 128), "bf16", "bf16", 16),
                                             ((7, 1, 128), "f16", "f32", 64), ((10, 2, 64), "bf16", "f32", 16)])
def test_prefill_tile_edges(gpu, heads, kv, act, bs):
    H, KH, hd = heads
    tile = 128 // (H // KH)
    q_len = [2, tile - 1, tile, tile + 1, 65, 7, 3, 1, 1]
    ctx = [2, tile - 1, tile + 62, tile + 64, 130, 64, 68, 40, 333]
    ctx = [max(a, b) for a, b in zip(ctx, q_len)]
    case = make_case(ctx, H, KH, hd, bs, q_len=q_len, seed=H, kv_bf16=kv == "bf16", kv_f16=kv == "f16")
    poison_unused(case)
    check(case, act, gpu, want_split=False)


# tiles split over partitions (their merge, of 2 to 16 partials), with XCD-local
# and with write-through partials, beside split decode rows
@pytest.mark.parametrize("flags", [0, LE_PLAN_XCD_LOCAL])
@pytest.mark.parametrize("heads,kv", [((14, 2, 64), "bf16"), ((8, 8, 128), "bf16"), ((32, 4, 64), "f16")])
def test_prefill_split_tiles(gpu, heads, kv, flags):
    H, KH, hd = heads
    case = make_case([577, 1500, 700, 6000, 1100, 2500], H, KH, hd, 16, q_len=[5, 40, 33, 3, 1, 1], seed=3,
                     kv_bf16=kv == "bf16", kv_f16=kv == "f16")
    check(case, "f32", gpu, want_split=True, flags=flags)


# partitions of more than 128 blocks (of 8 keys): the tile reads its ids from
# the step's tables, in a step with decode rows and without
@pytest.mark.parametrize("decode", [False, True])
@pytest.mark.parametrize("kv", ["bf16", "f32"])
def test_prefill_ids_from_the_tables(gpu, kv, decode):
    ctx, q_len = [17600, 300] + [700, 30] * decode, [21, 40] + [1, 1] * decode
    case = make_case(ctx, 14, 2, 64, 8, q_len=q_len, seed=8, kv_bf16=kv == "bf16")
    plan = run_ragged(case, torch.float32, gpu)[2]
    P = plan.plan
    items = plan.host.numpy()[P.off_chunk_items:][:36 * P.n_chunk_items].view(np.int32).reshape(-1, 9)
    assert (items[:, 6] < 0).any() and (items[items[:, 1] > 0, 6] >= 0).any()

    def bar(qh, want):  # twice the error of the 32-row tiles, which make the same roundings, and an ulp
        old = run_ragged(case, torch.float32, gpu, chunk_q_tile=32)[0]
        return 2 * max_abs(old, want) + 2.0 ** -22 * float(np.nanmax(np.abs(want)))

    check(case, "f32", gpu, want_split=True, bar=bar)


# Steps that the planner splits though they need no workspace: with a null or a
# short workspace their rows and tiles run whole, like the undivided rows of the
# 32-row plan; a step that needs one is refused as before.
@pytest.mark.parametrize("heads,kv,ctx,q_len", [
    ((32, 8, 128), "bf16", [1500, 2000, 84, 140, 30], [1, 1, 17, 40, 1]), ((14, 2, 64), "f16", [300, 1900, 9], [300, 1, 3]),
    ((14, 2, 64), "f32", [341], [341]), ((16, 16, 64), "f32", [200, 1400, 300], [132, 1, 50]),
    ((28, 4, 128), "f32", [640, 500, 257, 1], [1, 1, 1, 1]), ((14, 2, 64), "f32", [600], [1])])
def test_steps_without_workspace_run_whole(gpu, heads, kv, ctx, q_len):
    import ctypes
    from llm_engine_amd import _lib, kernels
    from gpu_util import device_q, slices_of, to_dev_cache
    H, KH, hd = heads
    case = make_case(ctx, H, KH, hd, 16, q_len=q_len, seed=len(ctx), kv_bf16=kv == "bf16", kv_f16=kv == "f16")
    poison_unused(case)
    q, qh = device_q(case, torch.float32, gpu)
    kc, vc = to_dev_cache(case.k_cache, gpu), to_dev_cache(case.v_cache, gpu)
    want = oracle_out(case, qh)
    tol = TOL_F32 if kv == "f32" else emulated_bar(case, qh, want)

    def run(plan, ws, nbytes):
        out = torch.full_like(q, float("nan"))
        st = _lib.load().le_ragged_paged_attention(
            q.data_ptr(), _lib.LE_F32, kc.data_ptr(), vc.data_ptr(), plan.plan.cfg.kv_dtype, kc.numel() // (16 * KH * hd),
            ctypes.byref(plan.plan), case.scale, out.data_ptr(), ws, nbytes, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        return st, out.cpu().numpy()

    for flags in (0, LE_PLAN_XCD_LOCAL):
        plan = kernels.Plan(slices_of(case), H, KH, hd, 16, kc.dtype, flags=flags).upload()
        assert plan.workspace_size() > 0 and plan.plan.cfg.chunk_partition_tokens == -1
        short = torch.zeros(4096, dtype=torch.uint8, device=gpu)
        (st, whole), (st2, again) = run(plan, None, 0), run(plan, short.data_ptr(), 4096)
        assert st == st2 == 0 and np.array_equal(whole, again) and not short.any()
        assert np.isfinite(whole).all() and np.abs(whole - want).max() <= tol
    split = kernels.Plan(slices_of(case), H, KH, hd, 16, kc.dtype, partition_tokens=16, chunk_q_tile=32).upload()
    assert run(split, None, 0)[0] == _lib.LE_ENOSPACE or split.workspace_size() == 0


@pytest.mark.parametrize("ctx", [[640, 500, 257, 1], [300]])
def test_store_without_workspace(gpu, ctx):
    """The store in the launch, rows run whole: the same bits as the store first and the attention after it, and the
    same cache."""
    import ctypes
    from llm_engine_amd import _lib, kernels
    from gpu_util import device_q, slices_of, to_dev_cache
    H, KH, hd = 28, 4, 128
    case = make_case(ctx, H, KH, hd, 16, seed=2)
    q, qh = device_q(case, torch.float32, gpu)
    plan = kernels.Plan(slices_of(case), H, KH, hd, 16, torch.float32).upload()
    assert plan.workspace_size() > 0 and plan.plan.cfg.chunk_partition_tokens == -1
    new = torch.randn(2, len(ctx), KH * hd, device=gpu, generator=torch.Generator(gpu).manual_seed(1))
    outs, caches = [], []
    for fused in (True, False):
        kc, vc = to_dev_cache(case.k_cache, gpu).clone(), to_dev_cache(case.v_cache, gpu).clone()
        out, nb = torch.full_like(q, float("nan")), kc.numel() // (16 * KH * hd)
        tail = (kc.data_ptr(), vc.data_ptr(), _lib.LE_F32, nb, ctypes.byref(plan.plan), case.scale, out.data_ptr(), None, 0,
                torch.cuda.current_stream().cuda_stream)
        if fused:
            st = _lib.load().le_ragged_paged_attention_store(q.data_ptr(), _lib.LE_F32, new[0].data_ptr(), new[1].data_ptr(),
                                                             _lib.LE_F32, *tail)
        else:
            kernels.store_kv(new[0], new[1], plan.dev_array("slots"), kc, vc)
            st = _lib.load().le_ragged_paged_attention(q.data_ptr(), _lib.LE_F32, *tail)
        torch.cuda.synchronize()
        assert st == 0
        outs.append(out.cpu().numpy())
        caches.append((kc.cpu().numpy(), vc.cpu().numpy()))
    assert np.array_equal(*outs) and all(np.array_equal(a, b) for a, b in zip(*caches))
    case.k_cache, case.v_cache = (c.reshape(d.shape) for c, d in zip(caches[0], (case.k_cache, case.v_cache)))
    assert max_abs(outs[0], oracle_out(case, qh)) <= TOL_F32


def tile32_bar(case, gpu, act="f32", **kw):
    """Twice the error of the 32-row tiles, which make the same roundings in another order."""
    def bar(qh, want):
        old, _, plan = run_ragged(case, ACT[act], gpu, chunk_q_tile=32, **kw)
        assert plan.plan.cfg.chunk_q_tile == 32
        err = np.abs(old.astype(np.float64) - want) - OUT_REL[act] * np.abs(want)
        return 2 * max(0.0, float(err.max()))
    return bar


def test_prefill_wide_tiles(gpu):
    """256-column tiles: a step past 1000 keys per workgroup slot."""
    case = make_case([16100, 15000], 32, 4, 64, 16, q_len=[300, 45], seed=4, kv_bf16=True)
    check(case, "f32", gpu, want_wide=True, want_split=True, bar=tile32_bar(case, gpu))


# wide tiles beside decode rows and alone, of both 16-bit cache types, with
# groups that fill the columns (8: 32 rows), leave some dead (7: 36 rows, 252
# columns) and have one row a column (1: 256 rows); split over partitions
# (few rows after many keys) and whole (three workgroups for every four slots)
@pytest.mark.parametrize("heads,kv,act,bs,ctx,q_len,decode", [
    ((32, 4, 64), "bf16", "bf16", 16, [16100, 15000], [300, 45], True), ((32, 4, 64), "f16", "f16", 16, [16100, 15000], [300, 45], True),
    ((32, 4, 64), "f16", "f32", 64, [16100, 15000], [300, 45], False),
    ((14, 2, 64), "bf16", "f32", 8, [17300, 9000], [560, 75], True), ((14, 2, 64), "f16", "bf16", 32, [17300, 9000], [560, 75], True),
    ((8, 8, 64), "bf16", "f32", 16, [15990, 12800], [1000, 300], True), ((8, 8, 64), "f16", "f32", 64, [15990, 12800], [1000, 300], True),
    ((8, 8, 64), "bf16", "bf16", 16, [15990, 12800], [1000, 300], False)])
def test_prefill_wide_split(gpu, heads, kv, act, bs, ctx, q_len, decode):
    H, KH, hd = heads
    ctx, q_len = ctx + [1200, 90] * decode, q_len + [1, 1] * decode
    case = make_case(ctx, H, KH, hd, bs, q_len=q_len, seed=H + bs, kv_bf16=kv == "bf16", kv_f16=kv == "f16")
    poison_unused(case)
    check(case, act, gpu, want_wide=True, want_split=True, bar=tile32_bar(case, gpu, act))


@pytest.mark.parametrize("kv,act,decode", [("bf16", "bf16", False), ("bf16", "f32", True), ("f16", "f16", True)])
def test_prefill_wide_whole(gpu, kv, act, decode):
    """Wide tiles that hold all keys of their rows: 54 tiles x 8 kv heads."""
    ctx, q_len = [3000, 2500] + [700, 3] * decode, [900, 800] + [1, 1] * decode
    case = make_case(ctx, 64, 8, 64, 16, q_len=q_len, seed=9, kv_bf16=kv == "bf16", kv_f16=kv == "f16")
    poison_unused(case)
    check(case, act, gpu, want_wide=True, want_split=False, bar=tile32_bar(case, gpu, act))


# Infinities and NaN: a key that scores -inf drops out, a row all of whose keys
# do is NaN; NaN or inf in a key, a value or a query row reaches the rows that
# attend to it. It reaches no other sequence, and of the chunk's earlier rows
# only, from a value (as 0 * NaN), those whose wave computes its 64-key tile: the
# rows of a wave (64 at most) and 63 before it. The 32-row tiles spread it over
# their 32 rows.
@pytest.mark.parametrize("kind", ["drop", "all", "nan_v", "inf_v", "inf_k", "nan_k", "nan_q"])
@pytest.mark.parametrize("heads,kv,wide", [((8, 2, 64), "bf16", False), ((8, 2, 64), "f16", False), ((3, 3, 64), "bf16", False),
                                           ((8, 2, 128), "bf16", False), ((14, 2, 64), "f32", False),
                                           ((3, 3, 64), "f32", False), ((32, 4, 64), "bf16", True)])
def test_prefill_nonfinite(gpu, heads, kv, wide, kind):
    H, KH, hd = heads
    ctx, q_len = [300, 150, 200, 40], [280, 60, 1, 40]
    if wide:
        ctx, q_len = ctx + [16300, 15000], q_len + [300, 45]
    case = make_case(ctx, H, KH, hd, 16, q_len=q_len, seed=11)
    at = {"nan_v": 191, "inf_v": 119}.get(kind, 150)  # a key of sequence 0's chunk
    slot = [case.blocks_of(s)[np.arange(ctx[s]) // 16].astype(np.int64) * 16 + np.arange(ctx[s]) % 16 for s in range(len(ctx))]
    k, v = case.k_cache.reshape(-1, KH, hd), case.v_cache.reshape(-1, KH, hd)
    q = case.q.reshape(-1, H, hd)
    if kind in ("drop", "all", "inf_k"):
        q[..., 0] = np.abs(q[..., 0]) + 1
    if kind in ("drop", "all"):
        k[slot[0][[3, 70, 150]] if kind == "drop" else slot[0][:40], :, 0] = -np.inf
    elif kind == "nan_v":
        v[slot[0][at], 0, 5] = np.nan
    elif kind == "inf_v":
        v[slot[0][at], 0, 5] = np.inf
    elif kind == "inf_k":
        k[slot[0][at], 0, 0] = np.inf
    elif kind == "nan_k":
        k[slot[0][at], 0, 0] = np.nan
    else:
        q[77, 1, 3] = np.nan
    if kv != "f32":
        case.k_cache, case.v_cache = ((oracle.f32_to_bf16(c) if kv == "bf16" else oracle.f32_to_f16(c)) for c in (case.k_cache, case.v_cache))
    new, _, plan = run_ragged(case, torch.float32, gpu)
    old = run_ragged(case, torch.float32, gpu, chunk_q_tile=32)[0]
    assert plan.plan.cfg.chunk_q_tile == (-1 if wide else 0)
    n, o = np.isfinite(new), np.isfinite(old)
    print(kind, "not finite: prefill", int((~n).sum()), "32-row", int((~o).sum()))
    far = (case.token_seq != 0) | (case.token_pos < at - 63 - (64 if wide else 32) // (H // KH))
    assert not (o & ~n)[far if kind in ("nan_v", "inf_v") else slice(None)].any()
    pos = case.token_pos
    seq0 = case.token_seq == 0
    must = {"drop": seq0 & (pos < 0), "all": seq0 & (pos < 40), "nan_q": np.arange(len(pos)) == 77}.get(kind, seq0 & (pos >= at))
    heads0 = n.reshape(len(pos), H, hd)[:, 1 if kind == "nan_q" else 0]
    if kv != "f32" or kind not in ("drop", "all"):  # (an infinity's terms: inf - inf)
        assert not heads0[must, 5].any() and n.reshape(len(pos), H, hd)[~seq0].all()
        assert kind != "drop" or n.all()
    both = n & o
    assert np.abs(new[both] - old[both]).max() <= (4e-6 if kv == "f32" else 0.03)


@pytest.mark.parametrize("kind", ["large", "negative", "rising"])
@pytest.mark.parametrize("hd,kv", [(64, "bf16"), (128, "bf16"), (64, "f16"), (128, "f16"), (64, "f32")])
def test_prefill_softmax_base(gpu, kind, hd, kv):
    """Scores far from 0 (the base that they are taken relative to starts at
    0): tens of log2 units wide, all far below 0, and rising along the keys so
    that the base moves tile after tile."""
    case = make_case([300, 150], 8, 2, hd, 16, q_len=[200, 33], seed=5)
    pos = np.zeros(case.k_cache.shape[0])
    for s in range(2):
        p = np.arange([300, 150][s])
        pos[case.blocks_of(s)[p // 16].astype(np.int64) * 16 + p % 16] = p
    k = case.k_cache.reshape(-1, 2, hd)
    q = case.q.reshape(-1, 8, hd)
    if kind == "large":
        k *= 8.0
    else:
        q[..., 0] = 8.0
        k[..., 0] = (-12.0 if kind == "negative" else pos[:, None] / 16)
    if kv == "f32":  # every product to fp32 rounding: the 32-row tiles' bar, and an ulp of the largest value
        bar = tile32_bar(case, gpu)
        check(case, "f32", gpu, bar=lambda qh, want: bar(qh, want) + 2.0 ** -22 * float(np.abs(case.v_cache).max()))
        return
    narrow = oracle.f32_to_bf16 if kv == "bf16" else oracle.f32_to_f16
    case.k_cache, case.v_cache = (narrow(c) for c in (case.k_cache, case.v_cache))
    check(case, "f32", gpu)


# fp32 caches of head_dim 64: every product to fp32 rounding. The bar is twice
# the error of the 32-row tiles, which make the same roundings in another order,
# and an ulp of the largest value for the order itself.
@pytest.mark.parametrize("flags", [0, LE_PLAN_XCD_LOCAL])
@pytest.mark.parametrize("heads,act,bs,split", [((14, 2, 64), "f32", 16, False), ((32, 4, 64), "bf16", 8, False),
                                                ((3, 3, 64), "f32", 32, False), ((14, 2, 64), "f32", 16, True),
                                                ((16, 16, 64), "f16", 64, True), ((8, 1, 64), "f32", 16, True)])
def test_prefill_f32_tiles(gpu, heads, act, bs, split, flags):
    H, KH, hd = heads
    tile = 128 // (H // KH)
    if split:
        q_len, ctx = [5, 40, tile + 1, 3, 2, 1, 1], [193, 1500, 700, 3000, 385, 1100, 2500]
    else:
        q_len, ctx = [2, tile - 1, tile, min(tile + 1, 130), 65, 7, 3, 1, 1], [2, 63, 64, 130, 128, 65, 68, 40, 333]
    ctx = [max(a, b) for a, b in zip(ctx, q_len)]
    case = make_case(ctx, H, KH, hd, bs, q_len=q_len, seed=H + bs)
    poison_unused(case)

    def bar(qh, want):
        old, _, plan = run_ragged(case, ACT[act], gpu, flags=flags, chunk_q_tile=32)
        assert plan.plan.cfg.chunk_q_tile == 32
        err = np.abs(old.astype(np.float64) - want) - OUT_REL[act] * np.abs(want)
        return 2 * max(0.0, float(err.max())) + 2.0 ** -22 * float(np.nanmax(np.abs(case.v_cache)))

    check(case, act, gpu, want_split=split, bar=bar, flags=flags)
