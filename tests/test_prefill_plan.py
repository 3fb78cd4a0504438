"""How a step's chunk rows are cut into prefill tiles (16-bit caches, and fp32
ones at head_dim 64; neither tile nor partition given): the work lists against the step, and against the
32-row tiles of the same step (chunk_q_tile given), over head groups, block
sizes, ragged rows, repeated sequences and step sizes."""
import numpy as np
import pytest
import torch

from llm_engine_amd import kernels
from llm_engine_amd._lib import LE_PLAN_TWO_LAUNCHES, LE_PLAN_XCD_LOCAL


def items_of(plan):
    P = plan.plan
    return plan.host.numpy()[P.off_chunk_items:P.off_chunk_items + 36 * P.n_chunk_items].view(np.int32).reshape(-1, 9)


def step(rng, bs, n_chunks, max_rows, max_hist, n_decode):
    out = []
    for i in range(n_chunks + n_decode):
        ln = int(rng.integers(2, max_rows + 1)) if i < n_chunks else 1
        start = int(rng.integers(0, max_hist + 1))
        nb = (start + ln + bs - 1) // bs
        out.append(kernels.Slice(i, start, ln, True, rng.permutation(nb + 3).astype(np.int32)[:nb],
                                 np.zeros(start + ln, np.int32)))
    return out


SHAPES = [(14, 2, 64), (32, 4, 64), (16, 16, 64), (32, 8, 128), (28, 4, 128), (6, 2, 64), (8, 1, 128)]


@pytest.mark.parametrize("heads", SHAPES)
@pytest.mark.parametrize("bs", [8, 16, 64, 512])
@pytest.mark.parametrize("kv", [torch.bfloat16, torch.float32])
def test_prefill_tiles_cover_the_step(heads, bs, kv):
    H, KH, hd = heads
    if kv == torch.float32 and hd != 64:
        pytest.skip("fp32 caches with head_dim 128 keep the 32-row tiles")
    rng = np.random.default_rng(H * 1000 + bs)
    wide = 0
    for n_chunks, max_rows, max_hist, n_decode in [(1, 2, 0, 0), (1, 40, 100, 3), (3, 300, 1500, 0), (2, 17, 9000, 5),
                                                   (8, 512, 1536, 0), (4, 600, 20000, 9), (1, 3, 16000, 0)]:
        sl = step(rng, bs, n_chunks, max_rows, max_hist, n_decode)

        def make(**kw):
            return kernels.Plan(sl, H, KH, hd, bs, kv, device="cpu", pin=False, **kw)

        plan, tiles32 = make(flags=LE_PLAN_XCD_LOCAL), make(flags=LE_PLAN_XCD_LOCAL, chunk_q_tile=32)
        P, old = plan.plan, tiles32.plan
        assert P.cfg.chunk_q_tile <= 0 and old.cfg.chunk_q_tile == 32
        is_wide = P.cfg.chunk_q_tile < 0
        wide += is_wide
        cols = 256 if is_wide else 128
        assert hd == 64 or not is_wide
        assert kv == torch.bfloat16 or not is_wide
        pos, tables = plan.host_array("positions"), plan.host_array("tables")
        toff, items = plan.host_array("table_offset"), items_of(plan)
        stride = P.decode_ids_stride
        n_ids = P.n_decode_items + P.n_chunk_items
        ids = plan.host.numpy()[P.off_decode_ids:P.off_decode_ids + 4 * n_ids * stride].view(np.int32).reshape(-1, stride)
        dec = plan.host.numpy()[P.off_decode_items:P.off_decode_items + 32 * P.n_decode_items].view(np.int32).reshape(-1, 8)
        dec_ids = max((int(d[4] - d[3]) for d in dec), default=0)
        by_tile, owned, bins = {}, [], {}
        for k, it in enumerate(items):
            tb, nq, b0, b1, p0, J, seq, part, live = (int(x) for x in it)
            if nq == 0:
                continue
            assert 1 <= nq * (H // KH) <= cols and (np.diff(pos[tb:tb + nq]) == 1).all()
            assert b1 > b0 and live == min((b1 - b0) * bs, pos[tb + nq - 1] + 1 - b0 * bs) and live >= 1
            row, n_ids, off = ids[P.n_decode_items + k], b1 - b0, toff[plan.host_array("token_seq")[tb]]
            if seq < 0:  # too many ids to list: the kernel reads them at tables + ~seq + b0
                assert ~seq == off and off + b1 <= P.n_table and n_ids > max(128, dec_ids)
                n_ids = 0
            assert (row[:n_ids] == tables[off + b0:off + b0 + n_ids]).all() and (row[n_ids:] == -1).all()
            by_tile.setdefault(tb, []).append((b0, b1, p0, J, part, nq))
            if J > 1:
                owned += [p0 + r * J for r in range(nq)]
                bins.setdefault(tb, set()).add(k % 8 if KH % 8 else 0)
            else:
                assert p0 == -1
        assert all(len(b) == 1 for b in bins.values())  # one tile's partitions on one XCD
        rows = set()
        for tb, parts in by_tile.items():
            parts.sort()
            nq = parts[0][5]
            assert parts[0][0] == 0 and parts[-1][1] == pos[tb + nq - 1] // bs + 1
            assert all(a[1] == b[0] for a, b in zip(parts, parts[1:])) and len(parts) == parts[0][3] <= 16
            assert [p[4] for p in parts] == list(range(len(parts)))
            rows |= set(range(tb, tb + nq))
        chunk_rows = sum(s.len for s in sl if s.len > 1)
        assert rows == set(range(chunk_rows))  # chunks first in these steps
        owned += [int(d[5]) for d in dec if d[5] >= 0]
        assert sorted(owned) == list(range(P.n_parts))
        # scratch: no more than the 32-row tiles take, or a small step's bound
        # (8 MiB for the tiles, 16 with an fp32 cache, and 5 MB for finer decode partitions)
        row_bytes = H * (hd * 4 + 8)
        small = (16 if kv == torch.float32 else 8) << 20
        assert P.n_parts * row_bytes <= max(old.n_parts * row_bytes, small) + 5_000_000
        assert P.n_parts * row_bytes <= max(old.n_parts * row_bytes, 31 << 20)
    assert wide > 0 or heads != (32, 4, 64) or kv == torch.float32  # both widths were seen


def test_prefill_tiles_only_where_asked_for_nothing():
    """Explicit sizes, the two-launch flag, fp32 caches with head_dim 128 and steps without
    arrival counters for every row keep the 32-row tiles; a plan's own
    resolved configuration gives the same plan again."""
    sl = step(np.random.default_rng(1), 16, 2, 400, 900, 3)

    def make(kv=torch.bfloat16, heads=(14, 2, 64), slices=sl, **kw):
        return kernels.Plan(slices, *heads, 16, kv, device="cpu", pin=False, **kw).plan

    auto = make()
    assert auto.cfg.chunk_q_tile <= 0 and auto.cfg.chunk_partition_tokens == 0
    again = make(chunk_q_tile=auto.cfg.chunk_q_tile, chunk_partition_tokens=auto.cfg.chunk_partition_tokens,
                 partition_tokens=auto.cfg.partition_tokens)
    assert (again.n_chunk_items, again.n_parts, again.bytes) == (auto.n_chunk_items, auto.n_parts, auto.bytes)
    for kw in (dict(chunk_q_tile=32), dict(chunk_q_tile=16), dict(chunk_partition_tokens=256),
               dict(flags=LE_PLAN_TWO_LAUNCHES), dict(kv=torch.float32, heads=(32, 8, 128))):
        assert make(**kw).cfg.chunk_q_tile in (16, 32)
    many = [kernels.Slice(i, 0, 600, True, np.arange(38, dtype=np.int32), np.zeros(600, np.int32)) for i in range(7)]
    assert make(heads=(16, 16, 64), slices=many).cfg.chunk_q_tile == 32  # 4200 rows x 16 kv heads
    assert make(heads=(16, 16, 64), slices=many[:6]).cfg.chunk_q_tile <= 0


def test_fp32_decode_partitions_of_a_small_step():
    """fp32 caches, decode rows only: the shortest partition from 256 keys on
    that leaves at most one workgroup a CU; the 16-bit rule (640 keys and more)
    where there is none."""
    rng = np.random.default_rng(12)
    seen = set()
    for trial in range(60):
        H, KH = [(14, 2), (32, 4), (32, 8), (16, 16)][trial % 4]
        lens = rng.integers(1, int(rng.choice([300, 1400, 5000])), size=int(rng.integers(1, 100)))
        sl = [kernels.Slice(i, int(n) - 1, 1, True, np.arange((n + 15) // 16, dtype=np.int32), np.zeros(int(n), np.int32))
              for i, n in enumerate(lens)]

        def make(kv):
            return kernels.Plan(sl, H, KH, 64, 16, kv, device="cpu", pin=False).plan

        def items(pt):
            return sum(-(-int(n) // pt) for n in lens)

        f32, b16 = make(torch.float32), make(torch.bfloat16)
        fits = [pt for pt in range(256, b16.cfg.partition_tokens, 128) if items(pt) * KH <= 256]
        assert f32.cfg.partition_tokens == (fits[0] if fits else b16.cfg.partition_tokens)
        assert f32.n_decode_items == items(f32.cfg.partition_tokens)
        seen.add(min(f32.cfg.partition_tokens, 640))
    assert {256, 640} <= seen


def plain_cut_splits(sl, H, KH, bs, partition=0):
    """Whether the plain cut (32-row tiles over 384 keys; decode rows over 640 keys, 2048 beside chunk rows, and more
    in steps of many keys) splits any row, that is, whether the step needs a workspace at all."""
    decode = [s.start + 1 for s in sl if s.len == 1]
    chunks = [s for s in sl if s.len > 1]
    part = -(-sum(decode) // max(1, 512 // KH))
    part = min(max(-(-part // 128) * 128, 2048 if chunks else 640), 4096) if partition == 0 else partition
    if partition == 0 and not chunks:
        while part < 4096 and sum(-(-n // part) for n in decode) * KH > 512:
            part += 128
    blocks = lambda n: -(-n // bs)
    return any(blocks(n) > blocks(part) for n in decode) or any(blocks(s.start + s.len) > blocks(384) for s in chunks)


@pytest.mark.parametrize("heads", SHAPES)
@pytest.mark.parametrize("kv", [torch.bfloat16, torch.float16, torch.float32])
def test_steps_without_workspace(heads, kv):
    """A step whose plain cut splits nothing needs no workspace, or its plan says that it may run whole without one,
    whatever finer partitions its cut takes: decode rows beside short chunks, fp32 prompts, fp32 decode rows. No other
    plan says so."""
    H, KH, hd = heads
    rng = np.random.default_rng(H + KH)
    seen = {True: 0, False: 0}
    for trial in range(120):
        bs = int(rng.choice([8, 16, 32, 64, 512]))
        n_chunks, n_decode = int(rng.integers(0, 5)), int(rng.integers(0, 30))
        max_rows, max_hist = int(rng.choice([10, 130, 380, 500])), int(rng.choice([0, 100, 600, 2040, 2500]))
        if n_chunks + n_decode == 0:
            continue
        sl = step(rng, bs, n_chunks, max_rows, max_hist, n_decode)
        for s in sl[:n_chunks]:  # chunks mostly within the plain cut's partition
            if trial % 3 and s.start + s.len > 384:
                s.start = max(0, 384 - s.len)
                s.blocks = s.blocks[:(s.start + s.len + bs - 1) // bs]
        partition = int(rng.choice([0, 0, 640, 2048]))
        plan = kernels.Plan(sl, H, KH, hd, bs, kv, device="cpu", pin=False, partition_tokens=partition)
        splits = plain_cut_splits(sl, H, KH, bs, partition)
        may_run_whole = plan.plan.cfg.chunk_partition_tokens == -1
        assert may_run_whole == (not splits and plan.workspace_size() > 0), (trial, [(s.start, s.len) for s in sl])
        seen[splits] += 1
    assert min(seen.values()) > 15


def test_plans_with_given_sizes_do_not_run_whole():
    """Explicit chunk tiles or partitions, two launches and fixed layouts: refused without their workspace as ever."""
    sl = [kernels.Slice(0, 0, 300, True, np.arange(19, dtype=np.int32), np.zeros(300, np.int32)),
          kernels.Slice(1, 1499, 1, True, np.arange(94, dtype=np.int32), np.zeros(1500, np.int32))]
    for kw in (dict(chunk_partition_tokens=128), dict(chunk_q_tile=32, partition_tokens=640),
               dict(flags=LE_PLAN_TWO_LAUNCHES, partition_tokens=640), dict(partition_tokens=640)):
        plan = kernels.Plan(sl, 14, 2, 64, 16, torch.bfloat16, device="cpu", pin=False, **kw)
        assert plan.workspace_size() > 0 and plan.plan.cfg.chunk_partition_tokens != -1, kw
    fixed = kernels.Plan(sl[1:], 14, 2, 64, 16, torch.float32, device="cpu", pin=False, partition_tokens=2048,
                         table_capacity=128)
    assert fixed.workspace_size() > 0 and fixed.plan.cfg.chunk_partition_tokens != -1


@pytest.mark.parametrize("bs", [8, 16])
@pytest.mark.parametrize("hist", [0, 2000, 16384])
def test_decode_ids_beside_prefill_tiles(bs, hist):
    """The decode items' block ids in a mixed step stay as many as the decode rows need, or 128, whatever the chunk's
    history: a tile over the whole of a long context does not widen their rows."""
    def plan(chunk):
        sl = [kernels.Slice(0, hist, 2048, True, np.arange((hist + 2048) // bs, dtype=np.int32),
                            np.zeros(hist + 2048, np.int32))] if chunk else []
        sl += [kernels.Slice(1 + i, 1023, 1, True, np.arange(1024 // bs, dtype=np.int32) + 7 * i,
                             np.zeros(1024, np.int32)) for i in range(64)]
        return kernels.Plan(sl, 32, 8, 128, bs, torch.bfloat16, device="cpu", pin=False, partition_tokens=1024)

    def ids(p):
        w = p.plan.decode_ids_stride
        return p.host.numpy()[p.plan.off_decode_ids:][:64 * 4 * w].view(np.int32).reshape(64, w)

    mixed, alone = plan(True), plan(False)
    P, n = mixed.plan, 1024 // bs
    assert P.cfg.chunk_q_tile == 0 and P.n_decode_items == alone.plan.n_decode_items == 64
    assert alone.plan.decode_ids_stride == n and P.decode_ids_stride <= max(n, 128)
    assert (ids(mixed)[:, :n] == ids(alone)).all() and (ids(mixed)[:, n:] == -1).all()
