"""GPU parity of the small-batch decode plans (VK_SCHED_AUTO): one workgroup per
(sequence, KV head), or partitions of a workgroup each and the merge launch, for
every KV type, q type and head width, at context lengths around a tile, a
wave's share and a partition; the append and the rotation folded in for the
plans that fold them. Pool bytes bit for bit and outputs within the stated
tolerance of the oracle (cases.tol_check; fp32 pools with fp32 q within
2e-5 + 2e-4 |ref|, the bound of tests/test_gpu_fp32_kv.py)."""
import numpy as np
import pytest

import pyoracle as O
import velokv
from cases import BS, make_case, oracle_layer, tol_check
from test_gpu_append_copy import assert_layer_equal, gpu_pool
from test_gpu_append_rope_decode import check, fused
from test_gpu_append_decode import oracle_layer_in
from test_gpu_head_dim_any import hd_case, gpu_pool as hd_pool, oracle_padded, oracle_decode

pytestmark = pytest.mark.gpu

# (lengths, whether the plan cuts them into partitions): alone and short; ragged with an
# empty context, tile edges and one long context; alone and long; one tile over a partition
LENS = [([1], False), ([129], False), ([0, 1, 16, 17, 31, 250, 255], False), ([5000], True),
        ([0, 15, 2049, 300, 4100, 1], True), ([2048, 2047, 2033, 2032], True)]


def plan(ctx, pool, case, qd, total=None):
    return ctx.decode_plan(pool, case.S, case.n_heads, int(case.ctx_lens.max()), bt_stride=case.block_tables.shape[1],
                           q_dtype=velokv.DT_F32 if qd == np.float32 else velokv.DT_F16,
                           sum_context_len=int(case.ctx_lens.sum()) if total is None else total)


def close(got, ref, kv, qd):
    if kv == O.F32 and qd == np.float32:
        assert np.all(np.abs(got - ref) <= 2e-5 + 2e-4 * np.abs(ref))
        return
    ok, err, nbad = tol_check(got, ref)
    assert ok, f"max err {err:.3g}, {nbad} out of tolerance"


@pytest.mark.parametrize("lens,parts", LENS)
@pytest.mark.parametrize("qd", [np.float16, np.float32])
@pytest.mark.parametrize("kv", [O.F32, O.F16, O.I8_REF, O.I8_BLK])
def test_decode(ctx, kv, qd, lens, parts):
    """Two KV heads, groups of 3; the sum of the lengths exact, unknown and wrong (it may only
    choose a plan): the same rows."""
    print(f"small decode kv={kv} q={np.dtype(qd).name} lens={lens}", flush=True)
    case = make_case(kv, np.maximum(lens, 1), n_kv_heads=2, n_heads=6, seed=3100 + len(lens), outlier_scale=8.0)
    pool, layer = gpu_pool(ctx, case), oracle_layer(case)
    case.ctx_lens = np.array(lens, np.int32)
    ref = O.paged_decode(layer, case.q.astype(qd), case.block_tables, case.ctx_lens)
    q, tab, cl = ctx.upload(case.q.astype(qd)), ctx.upload(case.block_tables), ctx.upload(case.ctx_lens)
    for total in (int(case.ctx_lens.sum()), 0, 7):
        pl = plan(ctx, pool, case, qd, total)
        assert total or len(lens) == 1 or pl["schedule"] == velokv.SCHED_STREAM, pl  # unknown lengths
        if not total and len(lens) > 1:
            continue
        assert pl["schedule"] == velokv.SCHED_WORKGROUP or max(lens) <= 64, pl
        assert not parts or (pl["max_partitions"] > 1 and pl["merge_launch"]), pl
        out = ctx.alloc(case.q.size * 4)
        ctx.paged_decode(pool, 0, q, velokv.DT_F32 if qd == np.float32 else velokv.DT_F16, out, cl, case.S, 6,
                         int(case.ctx_lens.max()), block_tables=tab, bt_stride=case.block_tables.shape[1],
                         sum_context_len=total)
        ctx.sync()
        close(out.download(case.q.shape, np.float32), ref, kv, qd)


@pytest.mark.parametrize("hd", [64, 96])
@pytest.mark.parametrize("lens", [[70, 1, 333], [4500]])
@pytest.mark.parametrize("kv", [O.F32, O.F16, O.I8_REF, O.I8_BLK])
def test_decode_other_head_dims(ctx, kv, lens, hd):
    print(f"small decode kv={kv} hd={hd} lens={lens}", flush=True)
    case = hd_case(kv, lens, hd, seed=3200 + hd)
    pool = hd_pool(ctx, case, hd)
    stride, top = case.block_tables.shape[1], int(case.ctx_lens.max())
    pl = ctx.decode_plan(pool, case.S, case.n_heads, top, bt_stride=stride, sum_context_len=int(case.ctx_lens.sum()))
    assert pl["schedule"] == velokv.SCHED_WORKGROUP, pl
    out = ctx.alloc(case.S * case.n_heads * hd * 4)
    ctx.paged_decode(pool, 0, ctx.upload(case.q), velokv.DT_F16, out, ctx.upload(case.ctx_lens), case.S, case.n_heads,
                     top, block_tables=ctx.upload(case.block_tables), bt_stride=stride,
                     sum_context_len=int(case.ctx_lens.sum()))
    ctx.sync()
    ref = oracle_decode(oracle_padded(case, hd), case.q, hd, case.block_tables, case.ctx_lens)
    close(out.download((case.S, case.n_heads, hd), np.float32), ref, kv, np.float16)


@pytest.mark.parametrize("lens", [[1], [16], [129], [5001], [17, 250, 1], [2049, 300, 4100, 16]])
@pytest.mark.parametrize("style", [0, O.ROPE_INTERLEAVED, O.ROPE_HALF])
@pytest.mark.parametrize("kv", [O.F32, O.F16, O.I8_REF, O.I8_BLK])
def test_append(ctx, kv, style, lens):
    """The new tokens appended (and rotated) by the decode launch where the plan folds them (one
    sequence of any type, ragged fp16 and any int8 block batch), else by a launch before it."""
    print(f"small append kv={kv} style={style} lens={lens}", flush=True)
    case = make_case(kv, lens, n_kv_heads=2, n_heads=8, seed=3300 + len(lens), outlier_scale=8.0)
    for qd in (np.float16, np.float32):
        if style:
            pl, pool, got, table, n_pos, ws = fused(ctx, case, style, qd, velokv.SCHED_AUTO)
            folds = len(lens) == 1 or kv in (O.F16, O.I8_BLK)
            assert pl["schedule"] != velokv.SCHED_WORKGROUP or (ws == 0) == folds, (pl, ws)
            check(ctx, case, style, qd, velokv.SCHED_AUTO, pl, pool, got, table, n_pos)
            continue
        pool = gpu_pool(ctx, case, with_last=False)
        sl, kk, vv = case.last_slots()
        out = ctx.alloc(case.q.size * 4)
        ctx.append_decode(pool, 0, ctx.upload(kk), ctx.upload(vv), velokv.DT_F16, ctx.upload(case.q.astype(qd)),
                          velokv.DT_F32 if qd == np.float32 else velokv.DT_F16, out, ctx.upload(case.ctx_lens), case.S, 8,
                          int(case.ctx_lens.max()), block_tables=ctx.upload(case.block_tables),
                          bt_stride=case.block_tables.shape[1], sum_context_len=int(case.ctx_lens.sum()))
        ctx.sync()
        ref = oracle_layer_in(case, np.float16)
        assert_layer_equal(pool, 0, ref)
        want = O.paged_decode(ref, case.q.astype(qd), case.block_tables, case.ctx_lens)
        close(out.download(case.q.shape, np.float32), want, kv, qd)


@pytest.mark.parametrize("first", [200, 208])  # the two tokens in one block, in two
@pytest.mark.parametrize("kv", [O.F32, O.F16, O.I8_REF, O.I8_BLK])
def test_append_of_one_sequence_twice(ctx, kv, first):
    """Two rows of the call on one table row at lengths L and L + 1: both tokens are stored before
    either row attends, so the second sees the first (uniform batches keep the append launch)."""
    print(f"small append of one sequence twice kv={kv} first={first}", flush=True)
    case = make_case(kv, [first], n_kv_heads=2, n_heads=8, seed=3400)
    pool = gpu_pool(ctx, case, with_last=False)
    r = np.random.default_rng(3401)
    k, v = (r.standard_normal((2, 2, 128)).astype(np.float16) for _ in range(2))
    q = r.standard_normal((2, 8, 128)).astype(np.float16)
    lens = np.array([first, first + 1], np.int32)
    bt = np.zeros((2, first // BS + 1), np.int32)
    bt[:, :case.block_tables.shape[1]] = case.block_tables
    if first % BS == 0:
        bt[:, -1] = next(b for b in range(case.n_blocks) if b not in case.block_tables)
    ref = oracle_layer(case, with_last=False)
    O.append(ref, k, v, np.array([bt[0, (n - 1) // BS] * BS + (n - 1) % BS for n in lens], np.int64))
    out = ctx.alloc(q.size * 4)
    ctx.append_decode(pool, 0, ctx.upload(k), ctx.upload(v), velokv.DT_F16, ctx.upload(q), velokv.DT_F16, out,
                      ctx.upload(lens), 2, 8, first + 1, block_tables=ctx.upload(bt), bt_stride=bt.shape[1],
                      sum_context_len=int(lens.sum()))
    ctx.sync()
    assert_layer_equal(pool, 0, ref)
    close(out.download(q.shape, np.float32), O.paged_decode(ref, q, bt, lens), kv, np.float16)


@pytest.mark.parametrize("kv,G", [(O.F16, 4), (O.F16, 7), (O.F32, 4), (O.I8_BLK, 4)])
def test_scratch_of_the_larger_plan(ctx, kv, G):
    """A uniform batch in partitions, with a buffer that only fixed partitions fit: it takes those.
    One byte less is refused."""
    print(f"small scratch kv={kv} G={G}", flush=True)
    case = make_case(kv, [1500, 1500], n_kv_heads=2, n_heads=2 * G, seed=3600)
    pool, layer = gpu_pool(ctx, case), oracle_layer(case)
    ref = O.paged_decode(layer, case.q, case.block_tables, case.ctx_lens)
    q, tab, cl = ctx.upload(case.q), ctx.upload(case.block_tables), ctx.upload(case.ctx_lens)
    stride, args = case.block_tables.shape[1], (case.S, case.n_heads, 1500)
    assert plan(ctx, pool, case, np.float16)["max_partitions"] > 1
    need = ctx.decode_workspace_bytes(pool, *args, stride, sum_context_len=3000)
    ctx.set_decode_schedule(velokv.SCHED_SPLIT)
    less = ctx.decode_workspace_bytes(pool, *args, stride, sum_context_len=3000)
    ctx.set_decode_schedule(velokv.SCHED_AUTO)
    out = ctx.alloc(case.q.size * 4)
    run = lambda size: ctx.paged_decode(pool, 0, q, velokv.DT_F16, out, cl, *args, block_tables=tab, bt_stride=stride,
                                        workspace=ctx.alloc(max(need, less)), workspace_bytes=size, sum_context_len=3000)
    for size in {need, less}:
        run(size)
        ctx.sync()
        close(out.download(case.q.shape, np.float32), ref, kv, np.float16)
    with pytest.raises(velokv._capi.VkError):
        run(min(need, less) - 1)


# one long context among many short ones: KV heads, lengths
SKEWED = [(8, [20000] + [200] * 39), (8, [10000] + [150] * 69), (8, [5000] + [60] * 199), (2, [40000] + [200] * 99)]


@pytest.mark.parametrize("shape", range(len(SKEWED)))
def test_skewed_batch(ctx, shape):
    """Every wave's range within the 256 blocks it can hold, and the append and the outputs right."""
    hkv, lens = SKEWED[shape]
    case = make_case(O.F16, lens, n_kv_heads=hkv, n_heads=hkv, seed=3500 + shape)
    q, cl, tab = ctx.upload(case.q), ctx.upload(case.ctx_lens), ctx.upload(case.block_tables)
    _, kk, vv = case.last_slots()
    for kv in (O.F32, O.F16, O.I8_REF, O.I8_BLK):
        print(f"small skewed kv={kv} {hkv} heads, {len(lens)} sequences, longest {lens[0]}", flush=True)
        case.kv_type = kv
        pool = gpu_pool(ctx, case, with_last=False)
        for total in (sum(lens), 7):
            pl = plan(ctx, pool, case, np.float16, total)
            assert pl["max_blocks_per_wave"] <= 256, pl
        out = ctx.alloc(case.q.size * 4)
        ctx.append_decode(pool, 0, ctx.upload(kk), ctx.upload(vv), velokv.DT_F16, q, velokv.DT_F16, out, cl, case.S, hkv,
                          lens[0], block_tables=tab, bt_stride=case.block_tables.shape[1], sum_context_len=sum(lens))
        ctx.sync()
        ref = oracle_layer_in(case, np.float16)
        assert_layer_equal(pool, 0, ref)
        want = O.paged_decode(ref, case.q, case.block_tables, case.ctx_lens)
        close(out.download(case.q.shape, np.float32), want, kv, np.float16)
