"""GPU parity of paged attention (reference-shaped entry and ragged plan)
against the CPU oracle (oracle.c, restating ops.h:87-111) on identical inputs.

Tolerances (|got - want| against the fp32 oracle, per element):
  * fp32 K/V: 4e-6 (decode rows: exact fp32 products; chunk rows: exact
    fp32 products at head_dim 128, three-term bf16 products at head_dim 64,
    each within a few fp32 roundings of the exact product; other summation
    orders; the largest error seen is 1.3e-6; the target bar is 1e-3);
  * bf16 K/V: twice the error of the host emulation of the kernels'
    roundings on the same case (tests/precision.py: q and the softmax
    weights rounded to bf16 for the MFMA; gpu_util.emulated_bar). The
    emulation matches the GPU's error closely (config 2: 1.66e-3 emulated,
    1.65e-3 measured; config 3: 5.6e-3 and 5.5e-3), and every bar stays
    inside the target 2e-2.
With bf16 activations the oracle is fed the same bf16-rounded q, and the
output's own rounding adds 2^-8 |want| (round to nearest bf16: 2^-9
relative, doubled for the error carried into it)."""
import numpy as np
import pytest
import torch

from cases import loguniform_ctx, make_case, make_shared_prefix_case
from gpu_util import device_q, emulated_bar, i32, max_abs, oracle_out, poison_unused, slices_of, to_dev_cache
from llm_engine_amd._lib import LE_F32, LE_PLAN_TWO_LAUNCHES, LE_PLAN_XCD_LOCAL

pytestmark = pytest.mark.gpu

TOL_F32 = 4e-6
OUT_REL = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8}


def within(got, want, tol, act=torch.float32) -> bool:
    """|got - want| <= tol + OUT_REL[act] * |want|, elementwise."""
    g, w = np.asarray(got, dtype=np.float64), np.asarray(want, dtype=np.float64)
    return bool(np.all(np.abs(g - w) <= tol + OUT_REL[act] * np.abs(w)))


def run_decode(case, act, dev):
    from llm_engine_amd import kernels
    q, qh = device_q(case, act, dev)
    kc, vc = to_dev_cache(case.k_cache, dev), to_dev_cache(case.v_cache, dev)
    out = kernels.attention_decode(q, kc, vc, i32(case.tables, dev), i32(case.table_offset, dev),
                                   i32(case.token_seq, dev), i32(case.token_pos, dev),
                                   case.q_heads, case.kv_heads, case.head_dim, case.block_size,
                                   case.scale)
    torch.cuda.synchronize()
    return out.float().cpu().numpy(), qh


def run_ragged(case, act, dev, **plan_kw):
    from llm_engine_amd import kernels
    q, qh = device_q(case, act, dev)
    kc, vc = to_dev_cache(case.k_cache, dev), to_dev_cache(case.v_cache, dev)
    plan = kernels.Plan(slices_of(case), case.q_heads, case.kv_heads, case.head_dim,
                        case.block_size, kc.dtype, **plan_kw).upload()
    out = kernels.ragged_paged_attention(q, kc, vc, plan, case.scale)
    torch.cuda.synchronize()
    return out.float().cpu().numpy(), qh, plan


def ran_on(plan, tile):
    """Whether the step's chunk rows (if any) ran on 32-row tiles (tile 32), or
    on the default's: prefill tiles, but for fp32 caches of head_dim 128."""
    P = plan.plan
    default32 = P.cfg.kv_dtype == LE_F32 and P.cfg.head_dim == 128
    return P.n_chunk_items == 0 or (P.cfg.chunk_q_tile == 32) == (tile == 32 or default32)


def tol_for(case, qh, want=None):
    """The bar for a case: TOL_F32 with an fp32 cache, else twice the
    emulated 16-bit error of this case."""
    if case.k_cache.dtype == np.float32:
        return TOL_F32
    return emulated_bar(case, qh, want)


@pytest.mark.parametrize("kv_bf16", [False, True])
def test_decode_target_shape_two_rounds(gpu, kv_bf16):
    """The 64 x 4096 target point at full size: 256 items x 2 kv heads =
    512 workgroups, the launch size that takes the unbounded-register decode
    kernel (two rounds of one workgroup per CU); below it the two-per-CU
    kernel runs (every other decode test)."""
    case = make_case([4096] * 64, num_blocks=32768, seed=7, kv_bf16=kv_bf16)
    got, qh, plan = run_ragged(case, torch.float32, gpu)
    assert plan.plan.n_decode_items * case.kv_heads >= 512
    want = oracle_out(case, qh)
    err = max_abs(got, want)
    print(f"target kv_bf16={kv_bf16}: items {plan.plan.n_decode_items} max|err|={err:.3e}")
    assert within(got, want, tol_for(case, qh))


@pytest.mark.parametrize("kv_bf16", [False, True])
@pytest.mark.parametrize("act", [torch.float32, torch.bfloat16])
def test_decode_config2_shape(gpu, kv_bf16, act):
    """Config 2 at full size: 64 seqs, ctx log-uniform in [64, 4096], tables
    from a 32768-block pool, Qwen2.5-0.5B GQA shape."""
    rng = np.random.default_rng(2)
    ctx = loguniform_ctx(rng, 64, 64, 4096)
    case = make_case(ctx, num_blocks=32768, seed=2, kv_bf16=kv_bf16)
    got, qh = run_decode(case, act, gpu)
    want = oracle_out(case, qh)
    err = max_abs(got, want)
    print(f"config2 kv_bf16={kv_bf16} act={act}: max|err|={err:.3e}")
    assert within(got, want, tol_for(case, qh), act)


@pytest.mark.parametrize("kv_bf16", [False, True])
def test_ragged_equals_reference_shaped(gpu, kv_bf16):
    rng = np.random.default_rng(5)
    ctx = loguniform_ctx(rng, 40, 1, 3000)
    case = make_case(ctx, num_blocks=8192, seed=5, kv_bf16=kv_bf16)
    a, qh = run_decode(case, torch.float32, gpu)
    b, _, plan = run_ragged(case, torch.float32, gpu)
    want = oracle_out(case, qh)
    tol = tol_for(case, qh)
    assert within(a, want, tol)
    assert within(b, want, tol)
    assert plan.plan.n_chunk_items == 0


@pytest.mark.parametrize("q_heads,kv_heads,head_dim", [(32, 4, 64), (8, 8, 64), (16, 2, 128), (4, 1, 128)])
@pytest.mark.parametrize("kv_bf16", [False, True])
def test_decode_other_shapes(gpu, q_heads, kv_heads, head_dim, kv_bf16):
    """GQA group 8 (TinyLlama), no grouping, head_dim 128."""
    rng = np.random.default_rng(q_heads * 100 + head_dim)
    ctx = loguniform_ctx(rng, 12, 1, 2500)
    case = make_case(ctx, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim,
                     num_blocks=4096, seed=7, kv_bf16=kv_bf16)
    got, qh = run_decode(case, torch.float32, gpu)
    assert within(got, oracle_out(case, qh), tol_for(case, qh))
    got2, _, _ = run_ragged(case, torch.float32, gpu)
    assert within(got2, oracle_out(case, qh), tol_for(case, qh))


@pytest.mark.parametrize("block_size", [8, 32, 64])
def test_decode_block_sizes(gpu, block_size):
    rng = np.random.default_rng(block_size)
    ctx = loguniform_ctx(rng, 10, 1, 2000)
    case = make_case(ctx, block_size=block_size, num_blocks=2048, seed=block_size)
    got, qh = run_decode(case, torch.float32, gpu)
    assert within(got, oracle_out(case, qh), TOL_F32)
    got2, _, _ = run_ragged(case, torch.float32, gpu)
    assert within(got2, oracle_out(case, qh), TOL_F32)


@pytest.mark.parametrize("kv_bf16", [False, True])
def test_decode_partition_over_table_segments(gpu, kv_bf16):
    """Partitions longer than the 1024 block ids a workgroup stages in LDS at
    once (here 2400 and 1900 blocks in one partition): the table is staged in
    segments. Also the reference-shaped launch over the same rows."""
    ctx = [38400, 30000, 700]
    case = make_case(ctx, num_blocks=4500, seed=71, kv_bf16=kv_bf16)
    got, qh, plan = run_ragged(case, torch.float32, gpu, partition_tokens=40000)
    want = oracle_out(case, qh)
    err = max_abs(got, want)
    print(f"segments kv_bf16={kv_bf16}: items {plan.plan.n_decode_items} max|err| {err:.3e}")
    assert plan.plan.n_decode_items == 3
    assert within(got, want, tol_for(case, qh))
    ref_shaped, _ = run_decode(case, torch.float32, gpu)
    assert within(ref_shaped, want, tol_for(case, qh))


def test_decode_edges(gpu):
    """pos 0 (one key), exact block multiples, one row past a boundary, and a
    long 8192 context (several 512-position LDS chunks in one workgroup)."""
    ctx = [1, 2, 15, 16, 17, 32, 33, 511, 512, 513, 8192]
    case = make_case(ctx, num_blocks=1024, seed=11)
    got, qh = run_decode(case, torch.float32, gpu)
    want = oracle_out(case, qh)
    assert within(got, want, TOL_F32)
    # one partition covering the whole context: exercises the chunked online rescale
    got2, _, plan = run_ragged(case, torch.float32, gpu, partition_tokens=16384)
    assert plan.plan.n_combine_items == 0
    assert within(got2, want, TOL_F32)
    # pos 0 attends to exactly one key: output equals that V row
    v0 = case.v_cache[case.blocks_of(0)[0] * 16, :64]
    assert max_abs(got[0, :64], v0) < 1e-6


@pytest.mark.parametrize("tile", [0, 32])
@pytest.mark.parametrize("kv_bf16", [False, True])
def test_chunk_rows_small(gpu, kv_bf16, tile):
    """Prefill chunks (causal inside the chunk, over a cached prefix) beside
    decode rows. bf16 K/V runs the MFMA chunk kernel, fp32 the decode kernel."""
    ctx = [40, 97, 160, 300, 64, 500]
    q_len = [1, 1, 64, 37, 64, 17]   # chunk at offsets 0, 263, 96, 483
    case = make_case(ctx, q_len=q_len, num_blocks=1024, seed=13, kv_bf16=kv_bf16)
    got, qh, plan = run_ragged(case, torch.float32, gpu, chunk_q_tile=tile)
    assert ran_on(plan, tile)
    want = oracle_out(case, qh)
    err = max_abs(got, want)
    print(f"chunk rows kv_bf16={kv_bf16}: items dec={plan.plan.n_decode_items} "
          f"chunk={plan.plan.n_chunk_items} max|err|={err:.3e}")
    assert plan.plan.n_chunk_items > 0  # chunk tiles with either cache type
    assert within(got, want, tol_for(case, qh))
    ref_shaped, _ = run_decode(case, torch.float32, gpu)
    assert within(ref_shaped, want, tol_for(case, qh))


@pytest.mark.parametrize("tile", [0, 32])
@pytest.mark.parametrize("act,kv_bf16,flags", [(torch.float32, True, 0), (torch.bfloat16, True, 0),
                                               (torch.float32, False, 0), (torch.float32, True, LE_PLAN_XCD_LOCAL),
                                               (torch.float32, False, LE_PLAN_XCD_LOCAL)])
def test_mixed_step_config3(gpu, act, kv_bf16, flags, tile):
    """Config 3: 32 decode rows (ctx U[256, 2048]) + 2 prefill chunks of 512
    at cached offsets 0 and 1024: 32 + 2 * 512 = 1056 ragged rows, with bf16
    K/V (16-bit MFMA chunk tiles) and fp32 K/V (three-term bf16 MFMA chunk
    tiles), with
    write-through partials and with the XCD-local exchange."""
    rng = np.random.default_rng(3)
    dec_ctx = rng.integers(256, 2049, size=32)
    ctx = [512, 1536] + list(dec_ctx)
    q_len = [512, 512] + [1] * 32
    case = make_case(ctx, q_len=q_len, num_blocks=16384, seed=3, kv_bf16=kv_bf16)
    got, qh, plan = run_ragged(case, act, gpu, flags=flags, chunk_q_tile=tile)
    assert plan.plan.n_tokens == 1056
    assert plan.plan.n_chunk_items > 0 and plan.plan.xcd_local == (flags != 0)
    assert ran_on(plan, tile)
    want = oracle_out(case, qh)
    err = max_abs(got, want)
    print(f"config3 act={act} kv_bf16={kv_bf16} flags={flags}: max|err|={err:.3e}")
    assert within(got, want, tol_for(case, qh), act)


@pytest.mark.parametrize("kv_bf16", [False, True])
@pytest.mark.parametrize("mixed", [False, True])
def test_config5_shared_prefix_full_contexts(gpu, kv_bf16, mixed):
    """Config 5's attention step at full size: 128 sequences whose tables
    start with the same 32 refcounted prefix blocks (a 512-token shared
    prefix) and go on in blocks of their own, contexts up to 8192 (four
    sequences at 8192, the rest 512 + U[64, 3300]), all in a fragmented
    16384-block pool. Decode rows only, or (mixed) with four sequences
    prefilling a 256-row chunk right after the shared prefix, whose causal
    rows read the shared blocks through the MFMA chunk tiles."""
    rng = np.random.default_rng(55)
    suffix = np.concatenate([[7680] * 4, rng.integers(64, 3301, size=124)])
    q_len = None
    if mixed:
        suffix[4:8] = 256
        q_len = np.ones(128, dtype=np.int64)
        q_len[4:8] = 256
    case = make_shared_prefix_case(suffix, q_len=q_len, seed=55, kv_bf16=kv_bf16)
    assert int(case.table_len.max()) == 512
    got, qh, plan = run_ragged(case, torch.float32, gpu)
    assert (plan.plan.n_chunk_items > 0) == mixed
    want = oracle_out(case, qh)
    err = max_abs(got, want)
    print(f"config5 full contexts kv_bf16={kv_bf16} mixed={mixed}: {case.n_tokens} rows, max|err|={err:.3e}")
    assert within(got, want, tol_for(case, qh))


def test_mixed_step_two_launches(gpu):
    """A mixed step runs as one launch by default; the LE_PLAN_TWO_LAUNCHES
    plan flag runs the chunk and decode kernels one after the other. Both against the
    oracle, on a step with split decode rows and split chunk tiles."""
    ctx = [900, 40, 2500, 1700, 300]
    q_len = [300, 40, 1, 1, 1]
    case = make_case(ctx, q_len=q_len, num_blocks=1024, seed=61, kv_bf16=True)
    want = None
    for two in (0, LE_PLAN_TWO_LAUNCHES):
        got, qh, plan = run_ragged(case, torch.float32, gpu, partition_tokens=640, flags=two)
        if want is None:
            want = oracle_out(case, qh)
        err = max_abs(got, want)
        print(f"two_launches={two}: chunk {plan.plan.n_chunk_items} decode {plan.plan.n_decode_items} "
              f"parts {plan.plan.n_parts} max|err| {err:.3e}")
        assert plan.plan.n_chunk_items > 0 and plan.plan.n_decode_items > 3
        assert within(got, want, tol_for(case, qh))


def test_split_chunk_partials_beyond_fp16_range(gpu):
    """Split chunk tiles of a bf16 cache carry fp16 partials, so the fp16
    range (the reference's own cache range) bounds them. With V scaled by
    2^20 (exact in bf16, |V| far past 65504), every output element must be
    either within the bar or not finite: an overflow is loud, never a wrong
    finite value. Rows whose partials stayed in range (decode rows, unsplit
    tiles) stay exact to the bar."""
    import dataclasses
    import oracle
    ctx = [900, 700, 1500, 300]
    q_len = [300, 1, 200, 1]
    base = make_case(ctx, q_len=q_len, num_blocks=1024, seed=83, kv_bf16=True)
    v = oracle.bf16_to_f32(base.v_cache) * np.float32(2.0 ** 20)
    case = dataclasses.replace(base, v_cache=oracle.f32_to_bf16(v))
    got, qh, plan = run_ragged(case, torch.float32, gpu, partition_tokens=256, chunk_partition_tokens=256)
    assert plan.plan.n_chunk_items > 0 and plan.plan.n_parts > 0
    want = oracle_out(case, qh)
    tol = tol_for(case, qh)
    ok = np.abs(got.astype(np.float64) - want) <= tol
    loud = ~np.isfinite(got)
    print(f"|V| up to {np.abs(v).max():.3g}: {int(loud.sum())} of {got.size} outputs not finite")
    assert bool(np.all(ok | loud))
    assert loud.any()  # the split tiles' partials did overflow
    decode = np.repeat(np.array([case.seq_qlen[s] == 1 for s in case.token_seq]), 1)
    assert bool(np.all(ok[decode]))


def test_workspace_reused_across_plans(gpu):
    """One workspace serves steps of different shapes (as the engine uses it):
    a step with few rows and many split partials, then a larger mixed step
    whose split chunk tiles need the arrival counters. The counters must not
    land on the first step's partials."""
    from llm_engine_amd import kernels
    a = make_case([4096, 3000, 2500], num_blocks=2048, seed=31, kv_bf16=True)
    b = make_case([600, 700, 650] + [300] * 40, q_len=[100, 90, 70] + [1] * 40, num_blocks=4096,
                  seed=32, kv_bf16=True)
    plans, need = [], 0
    for case, part in ((a, 256), (b, 0)):
        q, qh = device_q(case, torch.float32, gpu)
        kc, vc = to_dev_cache(case.k_cache, gpu), to_dev_cache(case.v_cache, gpu)
        plan = kernels.Plan(slices_of(case), case.q_heads, case.kv_heads, case.head_dim,
                            case.block_size, kc.dtype, partition_tokens=part).upload()
        plans.append((case, q, qh, kc, vc, plan))
        need = max(need, plan.workspace_size())
    ws = kernels.new_workspace(need, gpu)
    for rep in range(2):
        for case, q, qh, kc, vc, plan in plans:
            assert plan.plan.n_parts > 0
            out = kernels.ragged_paged_attention(q, kc, vc, plan, case.scale, workspace=ws)
            torch.cuda.synchronize()
            err = max_abs(out.float().cpu().numpy(), oracle_out(case, qh))
            print(f"rep {rep} rows {plan.plan.n_tokens} parts {plan.plan.n_parts} "
                  f"chunk items {plan.plan.n_chunk_items}: max|err| {err:.3e}")
            assert within(out.float().cpu().numpy(), oracle_out(case, qh), tol_for(case, qh))
    assert int(ws[:512 * 1024].count_nonzero().item()) == 0  # counters left at zero


@pytest.mark.parametrize("tile", [0, 32])
@pytest.mark.parametrize("q_heads,kv_heads,head_dim", [(32, 4, 64), (8, 8, 64), (16, 2, 128), (4, 1, 128)])
def test_chunk_rows_other_shapes(gpu, q_heads, kv_heads, head_dim, tile):
    """The MFMA chunk kernels (prefill and 32-row tiles) beyond the Qwen shape: GQA group 8 and 1,
    head_dim 128, with partial row tiles, split tiles (merged in-kernel) and a
    cached prefix; bf16 K/V against the oracle."""
    ctx = [700, 333, 90, 1]
    q_len = [45, 333, 17, 1]  # chunk at offset 655, a whole-prompt chunk, a short tail, a decode row
    case = make_case(ctx, q_len=q_len, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim,
                     num_blocks=512, seed=41, kv_bf16=True)
    got, qh, plan = run_ragged(case, torch.float32, gpu, chunk_q_tile=tile)
    assert ran_on(plan, tile)
    want = oracle_out(case, qh)
    err = max_abs(got, want)
    print(f"chunk {q_heads}/{kv_heads}x{head_dim}: items {plan.plan.n_chunk_items} parts {plan.plan.n_parts} "
          f"max|err| {err:.3e}")
    assert plan.plan.n_chunk_items > 0 and plan.plan.n_parts > 0
    assert within(got, want, tol_for(case, qh))


@pytest.mark.parametrize("tile", [0, 32])
@pytest.mark.parametrize("block_size", [8, 32, 64])
def test_chunk_rows_block_sizes(gpu, block_size, tile):
    """Chunk rows and decode rows (one long enough to be split) in one step, so
    in one launch, at block sizes other than 16."""
    ctx = [600, 129, 64, 2000, 37]
    q_len = [100, 129, 3, 1, 1]
    case = make_case(ctx, q_len=q_len, block_size=block_size, num_blocks=512, seed=43, kv_bf16=True)
    got, qh, plan = run_ragged(case, torch.bfloat16, gpu, partition_tokens=512, chunk_q_tile=tile)
    assert ran_on(plan, tile)
    want = oracle_out(case, qh)
    err = max_abs(got, want)
    print(f"chunk block {block_size}: items chunk {plan.plan.n_chunk_items} decode {plan.plan.n_decode_items} "
          f"max|err| {err:.3e}")
    assert plan.plan.n_chunk_items > 0 and plan.plan.n_decode_items > 2
    assert within(got, want, tol_for(case, qh), torch.bfloat16)


def test_more_rows_than_arrival_counters(gpu):
    """A step with more (row, kv head) pairs than a workspace has arrival
    counters (65536) runs on 32-row tiles, if no row is split."""
    case = make_case([380] * 11, q_len=[380] * 11, q_heads=16, kv_heads=16, num_blocks=300, seed=71, kv_bf16=True)
    got, qh, plan = run_ragged(case, torch.bfloat16, gpu)
    assert plan.plan.n_tokens * 16 > 65536 and plan.plan.cfg.chunk_q_tile == 32 and plan.workspace_size() == 0
    want = oracle_out(case, qh)
    assert within(got, want, tol_for(case, qh), torch.bfloat16)


def test_chunk_tile16_and_long_context(gpu):
    """16-row chunk tiles (plan option), and a chunk over a 9000-token prefix:
    longer partitions (several LDS stages per item) keep a tile's split count
    within what the in-kernel merge stages."""
    ctx = [9000 + 40, 300]
    q_len = [40, 300]
    case = make_case(ctx, q_len=q_len, num_blocks=1024, seed=47, kv_bf16=True)
    for tile in (16, 32):
        got, qh, plan = run_ragged(case, torch.float32, gpu, chunk_q_tile=tile)
        want = oracle_out(case, qh)
        err = max_abs(got, want)
        print(f"tile {tile}: items {plan.plan.n_chunk_items} parts {plan.plan.n_parts} max|err| {err:.3e}")
        assert within(got, want, tol_for(case, qh))


@pytest.mark.parametrize("kv_bf16,new_bf16", [(True, False), (True, True), (False, False)])
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("part", [256, 0])
def test_store_then_attend(gpu, kv_bf16, new_bf16, mixed, part):
    """le_ragged_paged_attention_store: the step's new K/V rows are stored at
    the plan's slots (inside the decode launch on a decode-only step) and
    attended to. Equal to the oracle's store_kv then attention: the caches
    bit-exact on every slot, the outputs within tolerance. Split rows put the
    new row in the last partition: with 256-token partitions the storing
    workgroup's first tiles hold the new key (loaded again after the store);
    with the planner's partitions (part 0: about 500 keys for the 1500- and
    2049-token rows) they do not, and stand."""
    import oracle
    from llm_engine_amd import kernels
    rng = np.random.default_rng(51)
    ctx = [1, 17, 300, 1500, 64, 2049] + ([600] if mixed else [])
    q_len = [1] * 6 + ([70] if mixed else [])
    case = make_case(ctx, q_len=q_len, num_blocks=1024, seed=52, kv_bf16=kv_bf16)
    n, kv_dim = len(case.token_pos), case.kv_heads * case.head_dim
    k_new = rng.standard_normal((n, kv_dim), dtype=np.float32)
    v_new = rng.standard_normal((n, kv_dim), dtype=np.float32)
    if new_bf16:
        k_new = oracle.bf16_to_f32(oracle.f32_to_bf16(k_new))
        v_new = oracle.bf16_to_f32(oracle.f32_to_bf16(v_new))
    slots = np.array([case.blocks_of(s)[p // 16] * 16 + p % 16 for s, p in zip(case.token_seq, case.token_pos)],
                     dtype=np.int32)
    want_k, want_v = case.k_cache.copy(), case.v_cache.copy()
    oracle.store_kv(k_new, v_new, slots, want_k, want_v)
    case.k_cache, case.v_cache = want_k, want_v  # the oracle attends over the stored rows
    q, qh = device_q(case, torch.float32, gpu)
    old_k = make_case(ctx, q_len=q_len, num_blocks=1024, seed=52, kv_bf16=kv_bf16)
    kc, vc = to_dev_cache(old_k.k_cache, gpu), to_dev_cache(old_k.v_cache, gpu)
    plan = kernels.Plan(slices_of(case), case.q_heads, case.kv_heads, case.head_dim, case.block_size,
                        kc.dtype, partition_tokens=part).upload()
    assert np.array_equal(plan.host_array("slots"), slots)
    nd = torch.bfloat16 if new_bf16 else torch.float32
    out = kernels.ragged_paged_attention(q, kc, vc, plan, case.scale,
                                         k_new=torch.from_numpy(k_new).to(gpu).to(nd),
                                         v_new=torch.from_numpy(v_new).to(gpu).to(nd))
    torch.cuda.synchronize()
    got_k = kc.cpu().view(torch.int16).numpy().view(np.uint16) if kv_bf16 else kc.cpu().numpy()
    got_v = vc.cpu().view(torch.int16).numpy().view(np.uint16) if kv_bf16 else vc.cpu().numpy()
    assert np.array_equal(got_k.view(np.uint8), want_k.view(np.uint8))
    assert np.array_equal(got_v.view(np.uint8), want_v.view(np.uint8))
    err = max_abs(out.float().cpu().numpy(), oracle_out(case, qh))
    print(f"store+attend kv_bf16={kv_bf16} new_bf16={new_bf16} mixed={mixed} part={part}: parts {plan.plan.n_parts} "
          f"max|err| {err:.3e}")
    assert within(out.float().cpu().numpy(), oracle_out(case, qh), tol_for(case, qh))


@pytest.mark.parametrize("tile", [0, 32])
@pytest.mark.parametrize("seed", range(16))
def test_random_ragged_steps(gpu, seed, tile):
    """Randomised mixed steps against the oracle: the number of sequences,
    their contexts and rows (decode rows, chunks at cached offsets, whole
    prompts), the GQA shape, head dim, block size, cache and activation
    dtypes, and the decode partition size all drawn from a seeded generator.
    Every launch shape the planner produces for such steps (one launch or
    decode only, split and unsplit rows and tiles) is reached across the
    seeds. Every cache row outside the live positions is NaN, so a tile
    variant that lets a dead row into a result fails here too."""
    rng = np.random.default_rng(1000 + seed)
    q_heads, kv_heads = [(14, 2), (32, 4), (8, 8), (16, 2), (4, 1), (28, 4)][rng.integers(6)]
    head_dim = int(rng.choice([64, 128]))
    block_size = int(rng.choice([8, 16, 32]))
    kv_bf16 = bool(rng.integers(2))
    act = torch.bfloat16 if rng.integers(2) else torch.float32
    n = int(rng.integers(1, 12))
    ctx = np.exp(rng.uniform(np.log(1), np.log(3000), size=n)).astype(np.int64) + 1
    q_len = np.ones(n, dtype=np.int64)
    for s in range(n):
        if rng.uniform() < 0.35:
            q_len[s] = int(rng.integers(1, ctx[s] + 1))
    need = int(((ctx + block_size - 1) // block_size).sum())
    case = make_case(ctx, q_len=q_len, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim,
                     block_size=block_size, num_blocks=need + 64, seed=seed, kv_bf16=kv_bf16)
    poison_unused(case)
    part = int(rng.choice([0, 256, 640, 2048]))
    flags = int(rng.choice([0, LE_PLAN_XCD_LOCAL]))
    got, qh, plan = run_ragged(case, act, gpu, partition_tokens=part, flags=flags, chunk_q_tile=tile)
    assert ran_on(plan, tile)
    want = oracle_out(case, qh)
    assert np.isfinite(got).all()
    err = max_abs(got, want)
    print(f"seed {seed}: {q_heads}/{kv_heads}x{head_dim} bs {block_size} kv_bf16 {kv_bf16} act {act} flags {flags} "
          f"rows {plan.plan.n_tokens} dec {plan.plan.n_decode_items} chunk {plan.plan.n_chunk_items} "
          f"parts {plan.plan.n_parts}: max|err| {err:.3e}")
    assert within(got, want, tol_for(case, qh), act)


@pytest.mark.parametrize("kv_bf16", [False, True])
def test_split_rows_merge_in_launch(gpu, kv_bf16):
    """Split decode rows (2..7 partitions each) merge inside the launch,
    through write-through partials and through one XCD's L2
    (LE_PLAN_XCD_LOCAL): against the oracle on a decode-only step and on a
    mixed step (chunk rows beside them), as one launch and as two
    (LE_PLAN_TWO_LAUNCHES)."""
    rng = np.random.default_rng(77)
    ctx = loguniform_ctx(rng, 24, 700, 4096)
    for q_len in (None, [1] * 23 + [64]):
        case = make_case(ctx, q_len=q_len, num_blocks=8192, seed=78, kv_bf16=kv_bf16)
        want = None
        shapes = (0,) if q_len is None else (0, LE_PLAN_TWO_LAUNCHES)
        for flags in shapes + tuple(f | LE_PLAN_XCD_LOCAL for f in shapes):
            got, qh, plan = run_ragged(case, torch.float32, gpu, partition_tokens=640, flags=flags)
            if want is None:
                want = oracle_out(case, qh)
            err = max_abs(got, want)
            print(f"flags={flags} mixed={q_len is not None}: parts {plan.plan.n_parts} "
                  f"decode items {plan.plan.n_decode_items} max|err| {err:.3e}")
            assert plan.plan.n_parts > 0
            assert within(got, want, tol_for(case, qh))


def test_graph_replays_match_eager(gpu):
    """The ragged attention captured in a HIP graph (plan upload not included)
    and replayed several times, with eager launches sharing the workspace in
    between: every replay equals the eager output bit for bit (partials merge
    in partition order whatever the arrival order), and the oracle within
    tolerance. The launch allocates and clears nothing, and its arrival
    counters reset themselves, so replays need no workspace reset."""
    from llm_engine_amd import kernels
    ctx = [2900, 40, 1800, 3500, 700, 1300]
    q_len = [1, 40, 1, 1, 96, 1]
    case = make_case(ctx, q_len=q_len, num_blocks=2048, seed=91, kv_bf16=True)
    q, qh = device_q(case, torch.float32, gpu)
    kc, vc = to_dev_cache(case.k_cache, gpu), to_dev_cache(case.v_cache, gpu)
    plan = kernels.Plan(slices_of(case), case.q_heads, case.kv_heads, case.head_dim, case.block_size,
                        kc.dtype, partition_tokens=640).upload()
    assert plan.plan.n_chunk_items > 0 and plan.plan.n_parts > 0
    ws = kernels.new_workspace(plan.workspace_size(), gpu)
    eager = kernels.ragged_paged_attention(q, kc, vc, plan, case.scale, workspace=ws)
    torch.cuda.synchronize()
    want = oracle_out(case, qh)
    assert within(eager.float().cpu().numpy(), want, tol_for(case, qh))
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    out = torch.empty_like(eager)
    with torch.cuda.stream(s):
        kernels.ragged_paged_attention(q, kc, vc, plan, case.scale, out=out, workspace=ws, stream=s)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            kernels.ragged_paged_attention(q, kc, vc, plan, case.scale, out=out, workspace=ws, stream=s)
    torch.cuda.synchronize()
    for rep in range(4):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), f"replay {rep} differs from the eager launch"
        again = kernels.ragged_paged_attention(q, kc, vc, plan, case.scale, workspace=ws)
        torch.cuda.synchronize()
        assert torch.equal(again, eager)


@pytest.mark.parametrize("tile", [0, 32])
@pytest.mark.parametrize("kv", ["f32", "bf16", "f16"])
def test_unused_cache_rows_never_read(gpu, kv, tile):
    """Dead keys of a tile (past a partition's or row's end) are read at a
    live key's address and masked: with every unused cache row NaN, decode
    rows (both entry points, split rows included) and a mixed step with
    prefill-chunk rows still match the oracle everywhere."""
    rng = np.random.default_rng(11)
    ctx = list(loguniform_ctx(rng, 24, 1, 3000)) + [700, 1333]
    q_len = [1] * 24 + [77, 300]
    for ql in (None, q_len):
        case = make_case(ctx, q_len=ql, num_blocks=4096, seed=11, kv_bf16=kv == "bf16", kv_f16=kv == "f16")
        poison_unused(case)
        b, qh, plan = run_ragged(case, torch.float32, gpu, chunk_q_tile=tile)
        assert ran_on(plan, tile)
        want = oracle_out(case, qh)
        assert np.isfinite(b).all()
        assert within(b, want, tol_for(case, qh))
        if ql is None:
            a, _ = run_decode(case, torch.float32, gpu)
            assert np.isfinite(a).all()
            assert within(a, want, tol_for(case, qh))


def test_fp32_chunk_rows_wide_range(gpu):
    """fp32 chunk tiles at head_dim 64 hold each operand as three bf16 terms
    (hi + mid + lo). With keys scaled up (sharp softmax rows, large scores)
    and values spread over six decades, the error against the fp32 oracle,
    relative to the largest |V|, stays at the fp32-rounding level, as with
    the exact fp32 MFMA tile of head_dim 128 on the same data."""
    errs = {}
    for hd in (64, 128):
        case = make_case([1024, 1536] + [700] * 4, q_len=[64, 96] + [1] * 4, num_blocks=512, seed=17,
                         head_dim=hd)
        rng = np.random.default_rng(5)
        case.k_cache *= np.float32(6.0)
        case.v_cache *= (10.0 ** rng.uniform(-3, 3, size=case.v_cache.shape)).astype(np.float32)
        got, qh, plan = run_ragged(case, torch.float32, gpu)
        assert plan.plan.n_chunk_items > 0
        want = oracle_out(case, qh)
        vmax = float(np.max(np.abs(case.v_cache)))
        errs[hd] = max_abs(got, want) / vmax
        print(f"fp32 chunk rows hd={hd}: max|err|/max|V| = {errs[hd]:.3e} (max|V| {vmax:.3g})")
    # measured: 1.7e-6 (three-term, head_dim 64) and 2.5e-6 (exact fp32 MFMA,
    # head_dim 128); the accumulation over up to 1536 keys sets both
    assert errs[64] < 5e-6
    assert errs[64] <= 2 * errs[128]
