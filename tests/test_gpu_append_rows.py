"""GPU parity of the append's paths, bit for bit against the oracle: blocks filled whole, runs that
start or end inside a block that holds tokens already, single tokens, runs the all-at-once path does
not take (padding inside, an order that is not ascending), V token pairs in and out of order, rows at
addresses aligned to four bytes only, int8 block scales at their extremes (zero, past fp16), and each
pattern both in a short call (a workgroup per token and head) and in a long one (rows), its last tokens."""
import numpy as np
import pytest

import pyoracle as O
import velokv
from cases import BS
from test_gpu_append_copy import assert_layer_equal

pytestmark = pytest.mark.gpu

HKV, N_BLOCKS = 2, 12


def tile_w(hd):
    return 64 if hd <= 64 else 128


def patterns():
    """(name, slots) of one call after positions 0..20 of block order 3, 7 are in the pool."""
    b = lambda blk, lo, hi: [blk * BS + i for i in range(lo, hi)]
    return {
        "whole": b(5, 0, 16) + b(1, 0, 16) + b(9, 0, 3),                      # a prompt of 35 tokens
        "grow": b(7, 5, 16) + b(2, 0, 16) + b(11, 0, 16) + b(0, 0, 1),        # continues a block
        "drafts": b(7, 5, 13) + b(4, 12, 16) + b(6, 0, 4) + b(8, 15, 16),     # 8-token drafts, one over two blocks
        "single": [7 * BS + 5, 4 * BS, 9 * BS + 15, 10 * BS + 2],
        "padding": [-1, 7 * BS + 5, -1, 7 * BS + 6, 2 * BS, -1, -1, 2 * BS + 1, 5 * BS, N_BLOCKS * BS, -1],
        "wrap": b(2, 8, 16) + b(2, 0, 8) + b(4, 14, 16) + [4 * BS + 13],        # goes on in a block filled to its end
        "order": [2 * BS + 1, 2 * BS, 2 * BS + 3, 2 * BS + 2, 6 * BS + 1, 6 * BS + 2, 6 * BS + 4],
        "contiguous": b(8, 0, 16) + b(9, 0, 16) + b(10, 0, 16) + b(11, 0, 16),  # 64 slots in a row from the call's start
    }


def rows(r, n, hd, dt, extreme):
    x = (r.standard_normal((n, HKV, hd)) * 2.0).astype(np.float32)
    x *= np.linspace(0.5, 2.5, 50)[np.arange(n) % 50][:, None, None]  # scales grow along the call
    if extreme:
        x[0::5] = 0.0                              # rows of zeros: scale 0
        x[1::7] *= 1e-7
        if dt == np.float32:
            x[3::6] *= 2e7                         # amax / 127 past fp16: an infinite scale
    return np.ascontiguousarray(x.astype(dt))


def upload_at(ctx, a, offset):
    """The array in device memory at an address `offset` bytes past an allocation's start."""
    buf = ctx.alloc(a.nbytes + 64)
    buf.upload(a, offset)
    return buf, buf.ptr + offset


@pytest.mark.parametrize("lead", [0, 1101])  # padding slots before the pattern
@pytest.mark.parametrize("name", list(patterns()))
@pytest.mark.parametrize("hd", [128, 64, 96, 40])
@pytest.mark.parametrize("kv", [O.F32, O.F16, O.I8_REF, O.I8_BLK])
def test_append_patterns(ctx, kv, hd, name, lead):
    print(f"append rows kv={kv} hd={hd} {name} lead={lead}", flush=True)
    slots = np.array([-1] * lead + patterns()[name], np.int64)
    for style, dt, extreme, off in ((0, np.float16, False, 0), (0, np.float32, True, 4), (O.ROPE_HALF, np.float16, False, 4),
                                    (O.ROPE_INTERLEAVED, np.float32, False, 0), (O.ROPE_HALF, np.float32, False, 0)):
        r = np.random.default_rng(4100 + hd + 7 * style)
        pool = velokv.Pool(ctx, 1, N_BLOCKS, BS, HKV, hd, kv)
        T = tile_w(hd)
        ref = O.Layer(N_BLOCKS, HKV, BS, T, kv)
        pad = lambda x: np.pad(x, ((0, 0), (0, 0), (0, T - hd)))
        before = np.array([3 * BS + i for i in range(16)] + [7 * BS + i for i in range(5)], np.int64)
        n, n_pos, heads = len(slots), 64, 5
        table = velokv.rope_table(n_pos, hd, 10000.0)
        for sl, ex in ((before, False), (slots, extreme)):
            k, v = rows(r, len(sl), hd, dt, ex), rows(r, len(sl), hd, dt, ex)
            code = velokv.DT_F32 if dt == np.float32 else velokv.DT_F16
            (kb, kp), (vb, vp) = upload_at(ctx, k, off), upload_at(ctx, v, off)
            if style and sl is slots:
                pos = r.integers(0, n_pos, n).astype(np.int32)
                pos[-1] = n_pos  # outside the table: skipped
                q = (r.standard_normal((n, heads, hd))).astype(dt)
                qb, qp = upload_at(ctx, q, off)
                ctx.append_rope(pool, 0, kp, vp, code, ctx.upload(pos), ctx.upload(sl), n, ctx.upload(table), n_pos, style,
                                q=qp, q_dtype=code, n_heads=heads)
                kr, qr = rotate(k, pos, style, table), rotate(q, pos, style, table)
                use = np.where(pos < n_pos, sl, -1)
                O.append(ref, pad(kr), pad(v.astype(np.float32)), use)
                got_q = qb.download(q.shape, q.dtype, offset=off)
                assert np.array_equal(got_q, qr.astype(dt)), "q"
            else:
                ctx.append(pool, 0, kp, vp, code, ctx.upload(sl), len(sl))
                O.append(ref, pad(k.astype(np.float32)), pad(v.astype(np.float32)), sl)
            ctx.sync()
        assert_layer_equal(pool, 0, ref)


def rotate(x, pos, style, table):
    """x [n, heads, hd] rotated in fp32, every product and sum rounded by itself; rows whose position is
    outside the table as they are."""
    y, hd = x.astype(np.float32), x.shape[-1]
    a, b = (slice(0, hd // 2), slice(hd // 2, hd)) if style == O.ROPE_HALF else (slice(0, hd, 2), slice(1, hd, 2))
    out = y.copy()
    for i, p in enumerate(pos):
        if 0 <= p < len(table):
            c, s = table[p, :, 0], table[p, :, 1]
            out[i][:, a] = y[i][:, a] * c - y[i][:, b] * s
            out[i][:, b] = y[i][:, a] * s + y[i][:, b] * c
    return out


@pytest.mark.parametrize("n,in_a_row", [(5000, False), (5000, True), (17000, True)])
@pytest.mark.parametrize("kv", [O.F16, O.I8_BLK])
def test_append_prompt_of_many_windows(ctx, kv, n, in_a_row):
    """A prompt longer than a window of 16 tokens per workgroup, from an offset inside a block, over
    scattered pages and over pages handed out in order (more than 64 slots in a row, as in large pages)."""
    print(f"append long prompt kv={kv} n={n} in_a_row={in_a_row}", flush=True)
    r = np.random.default_rng(4200)
    blocks = (7 + n) // BS + 10
    perm = np.arange(blocks) if in_a_row else r.permutation(blocks)
    p = np.arange(7, 7 + n)
    sl = (perm[p // BS] * BS + p % BS).astype(np.int64)
    pool = velokv.Pool(ctx, 1, blocks, BS, HKV, 128, kv)
    ref = O.Layer(blocks, HKV, BS, 128, kv)
    k, v = ((r.standard_normal((n, HKV, 128)) * 3).astype(np.float16) for _ in range(2))
    ctx.append(pool, 0, ctx.upload(k), ctx.upload(v), velokv.DT_F16, ctx.upload(sl), n)
    ctx.sync()
    O.append(ref, k, v, sl)
    assert_layer_equal(pool, 0, ref)


def test_append_nan_scale(ctx):
    """A per-token int8 row of 128 NaN has the scale NaN, and of fewer dims (the tile's others are zeros)
    0, in a short call (a workgroup per token) as in a long one (rows); its codes are 0 (parity unpinned)."""
    for hd, want in ((128, np.nan), (96, 0.0), (64, 0.0)):
        for lead in (0, 1101):
            print(f"append NaN rows hd={hd} lead={lead}", flush=True)
            pool = velokv.Pool(ctx, 1, 2, BS, HKV, hd, O.I8_REF)
            k = np.full((lead + 1, HKV, hd), np.nan, np.float32)
            ctx.append(pool, 0, ctx.upload(k), ctx.upload(k), velokv.DT_F32, ctx.upload(np.array([-1] * lead + [BS], np.int64)),
                       lead + 1)
            ctx.sync()
            got = pool.download_layer(0)
            for key in ("ks", "vs"):
                scale = got[key].view(np.float32).reshape(2, HKV, BS)[1, :, 0]
                assert np.array_equal(scale, np.full(HKV, want, np.float32), equal_nan=True), (key, scale)
            assert not got["k"].any() and not got["v"].any()


def test_append_f16_bits(ctx):
    """fp16 rows go into an fp16 pool of 128 dims bit for bit, signalling NaN included, V pairs and single
    tokens, in a short call as in a long one; unrotated K rows do, and V rows whatever K does."""
    r = np.random.default_rng(4300)
    n, N = 3, 3 * HKV * 128
    where = np.arange(1, N + 1).reshape(n, HKV, 128).astype(np.float16)  # (integers: exact in fp16)
    slots = np.array([BS + 4, BS + 5, 7], np.int64)
    at = O.Layer(2, HKV, BS, 128, O.F16)
    O.append(at, where, where, slots)
    bits = r.integers(0, 1 << 16, N + 1).astype(np.uint16)
    bits[1:40] = np.arange(0x7C01, 0x7C01 + 39)  # signalling NaN
    bits[0] = 0
    rows16 = bits[where.astype(np.int64)]
    for lead in (0, 1101):
        for rope in (False, True):
            print(f"append fp16 bits lead={lead} rope={rope}", flush=True)
            pool = velokv.Pool(ctx, 1, 2, BS, HKV, 128, O.F16)
            x = ctx.upload(np.concatenate([np.zeros((lead, HKV, 128), np.uint16), rows16]))
            sl = ctx.upload(np.concatenate([np.full(lead, -1, np.int64), slots]))
            if rope:
                ctx.append_rope(pool, 0, x, x, velokv.DT_F16, ctx.upload(np.zeros(lead + n, np.int32)), sl, lead + n,
                                ctx.upload(velokv.rope_table(4, 128, 10000.0)), 4, O.ROPE_HALF)
            else:
                ctx.append(pool, 0, x, x, velokv.DT_F16, sl, lead + n)
            ctx.sync()
            got = pool.download_layer(0)
            for key in ("v",) if rope else ("k", "v"):
                ref = bits[np.frombuffer(getattr(at, key).tobytes(), np.float16).astype(np.int64)]
                assert np.array_equal(got[key].view(np.uint16), ref), key


def test_append_of_more_threads_than_a_grid_dimension(ctx):
    """17 M padding tokens and three real ones at the end: 34 M workgroups of 128 threads, where HIP
    takes less than 2^32 threads in one dimension of a grid."""
    kv, hkv, hd, n = O.F16, 8, 8, 17_000_000
    print(f"append of {n} tokens", flush=True)
    slots = np.full(n, -1, np.int64)
    slots[-3:] = [BS + 4, BS + 5, 7]
    r = np.random.default_rng(4400)
    tail = r.standard_normal((3, hkv, hd)).astype(np.float16)
    rows_in = ctx.alloc(n * hkv * hd * 2)  # (padding rows are read as they are and not stored)
    rows_in.upload(tail, (n - 3) * hkv * hd * 2)
    pool = velokv.Pool(ctx, 1, 2, BS, hkv, hd, kv)
    ctx.append(pool, 0, rows_in, rows_in, velokv.DT_F16, ctx.upload(slots), n)
    ctx.sync()
    ref = O.Layer(2, hkv, BS, 64, kv)
    x = np.pad(tail, ((0, 0), (0, 0), (0, 64 - hd)))
    O.append(ref, x, x, slots[-3:])
    assert_layer_equal(pool, 0, ref)
