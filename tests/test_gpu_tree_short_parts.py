"""Tree-verify calls of few units take partitions of less than 256 tokens; parity with the
oracle at the edges of that rule, and with a buffer that only the longer partitions fit."""
import numpy as np
import pytest

import pyoracle as O
import velokv
from cases import HD, oracle_layer
from test_gpu_append_copy import gpu_pool
from test_gpu_tree import check, mask_222, tree_case, tree_q

pytestmark = pytest.mark.gpu

SHAPES = [  # committed lengths, nodes, partition on 256 CUs: 8 KV heads, one 16- or 32-row tile each
    ([248], 8, 256),                  # one partition covers it: stays whole
    ([249], 8, 64),
    ([1, 63, 64, 3000], 8, 96),       # 4 x 8 heads x 47 units of 64 tokens are more than one a SIMD
    ([0, 2056, 255, 512, 4000], 8, 192),
    ([700, 5] * 8, 8, 96),
    ([1500] * 12, 8, 192),
    ([1600] * 15, 8, 256),            # past one unit a SIMD
]


def _run(ctx, pool, case, q, committed, mask, **kw):
    out = ctx.alloc(q.size * 4)
    ctx.tree_verify(pool, 0, ctx.upload(q), velokv.DT_F16, out, ctx.upload(np.asarray(committed, np.int32)),
                    ctx.upload(np.ascontiguousarray(mask, np.uint32)), case.S, q.shape[1], case.n_heads, max(committed),
                    block_tables=ctx.upload(case.block_tables), bt_stride=case.block_tables.shape[1], **kw)
    ctx.sync()
    return out.download((case.S, q.shape[1], case.n_heads, HD), np.float32)


@pytest.mark.parametrize("kv", [O.F32, O.F16, O.I8_REF, O.I8_BLK])
@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_short_partitions(ctx, kv, shape):
    committed, n, part = SHAPES[shape]
    print(f"tree short partitions kv={kv} committed={committed[:5]} n={n}", flush=True)
    case = tree_case(kv, committed, n, seed=71 + shape)
    ref_layer = oracle_layer(case)
    pool = gpu_pool(ctx, case)
    q = tree_q(case.S, n, case.n_heads, 7100 + shape)
    mask = np.tile(mask_222(n), (case.S, 1))
    stride = case.block_tables.shape[1]
    pl = ctx.tree_plan(pool, case.S, n, case.n_heads, max(committed), bt_stride=stride)
    assert pl["partition_tokens"] == part, pl
    ref = O.tree_verify(ref_layer, q, case.block_tables, committed, mask)
    check(_run(ctx, pool, case, q, committed, mask), ref, "short partitions")
    if part == 256:
        return
    need = ctx.tree_workspace_bytes(pool, case.S, n, case.n_heads, max(committed), stride)
    less = ctx.tree_workspace_bytes(pool, case.S, n, case.n_heads, max(committed), stride, partition_tokens=256)
    assert less < need
    for size in (need, need - 1, less):
        ws = ctx.alloc(size)
        check(_run(ctx, pool, case, q, committed, mask, workspace=ws, workspace_bytes=size), ref, f"workspace {size}")
    with pytest.raises(velokv._capi.VkError):
        _run(ctx, pool, case, q, committed, mask, workspace=ws, workspace_bytes=less - 1)
