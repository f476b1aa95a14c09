"""Performance cases of the KV-cache hot path: what a serving program calls, at the sizes it calls it with.

Four kinds of work, each through velokv's public entry points:

  step     one layer of a decode step: rope, append of every sequence's new token and paged decode
           attention over the context with it (Context.append_rope_decode / append_decode)
  prompt   one layer of a prompt's KV write: rope of q and K and the append of all its tokens
           (Context.append_rope)
  verify   a speculative step: the shared partial block's copy-on-write copy, then in each layer the
           append of the draft tokens and tree-verify attention, then the commit of the accepted
           path in all layers (Context.copy_blocks, append, tree_verify, tree_commit)
  handoff  prefill to decode migration: sequences' pages packed into NIXL wire records and unpacked
           into another pool (Context.nixl_pack, nixl_unpack)

listed() names twelve, draw() gives others of the same ranges. Lengths follow from a case's sizes,
everything else from the seed.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "velo-core_amd"))
import velokv  # noqa: E402

KV_TYPES = {"fp32": velokv.KV_F32, "fp16": velokv.KV_F16, "int8": velokv.KV_I8_REF, "int8blk": velokv.KV_I8_BLK}
CODE_BYTES = {"fp32": 4, "fp16": 2, "int8": 1, "int8blk": 1}
STYLES = {"half": velokv.ROPE_HALF, "interleaved": velokv.ROPE_INTERLEAVED}
TILE = 16  # tokens of a storage tile, and of an int8blk scale
ROPE_BASE = 10000.0


def listed():
    return [
        # one user, a short chat: launches and latency
        _step("step_1x512_fp16", 1, 512, 512, 32, 8, 128, "fp16", "fp16", 16, "half"),
        # a few users of a compressed cache, odd lengths
        _step("step_4x600-3000_int8blk", 4, 600, 3000, 32, 8, 128, "int8blk", "fp16", 16, "half"),
        # the default cache type with fp32 activations, a small server
        _step("step_8x100-2500_fp32", 8, 100, 2500, 32, 8, 128, "fp32", "fp32", 16, "interleaved"),
        # a small model: 64-dim heads, 7 query heads per KV head, per-token scales, 64-token pages
        _step("step_24x64-1500_int8_d64", 24, 64, 1500, 14, 2, 64, "int8", "fp32", 64, "half"),
        # a full ragged batch over the compressed cache
        _step("step_64x1024-8192_int8blk", 64, 1024, 8192, 32, 8, 128, "int8blk", "fp16", 16, "none"),
        # a full uniform batch over an fp16 cache
        _step("step_64x8192_fp16", 64, 8192, 8192, 32, 8, 128, "fp16", "fp16", 16, "none"),
        # one GPU's share of a long-context batch of a 70B-shaped model: the largest call
        _step("step_32x32768_int8blk_gqa8", 32, 32768, 32768, 64, 8, 128, "int8blk", "fp16", 16, "half"),
        # one prompt of ordinary length
        _prompt("prompt_1x777_fp16", 1, 777, 777, 32, 8, 128, "fp16", "fp16", 16, "half"),
        # a batch of prompts into the compressed cache
        _prompt("prompt_4x1500-2500_int8blk", 4, 1500, 2500, 32, 8, 128, "int8blk", "fp16", 16, "half"),
        # speculative decoding of a few users, no shared prefix
        _verify("verify_6x200-3000_fp16", 6, 0, 200, 3000, 13, 2, 32, 8, 128, "fp16", "fp16"),
        # speculative decoding of a full batch behind one shared system prompt
        _verify("verify_256_shared4096_int8blk", 256, 4096, 0, 512, 8, 2, 32, 8, 128, "int8blk", "fp16"),
        # four long sequences moved from a prefill to a decode pool
        _handoff("handoff_4x2000-4000_int8blk", 4, 2000, 4000, 8, 8, 128, "int8blk"),
    ]


def _step(name, seqs, lo, hi, heads, kv_heads, dim, kv, act, page, rope):
    return dict(name=name, kind="step", seqs=seqs, lo=lo, hi=hi, heads=heads, kv_heads=kv_heads, dim=dim, kv=kv,
                act=act, page=page, rope=rope)


def _prompt(name, seqs, lo, hi, heads, kv_heads, dim, kv, act, page, rope):
    return dict(_step(name, seqs, lo, hi, heads, kv_heads, dim, kv, act, page, rope), kind="prompt")


def _verify(name, seqs, prefix, lo, hi, nodes, layers, heads, kv_heads, dim, kv, act):
    return dict(name=name, kind="verify", seqs=seqs, prefix=prefix, lo=lo, hi=hi, nodes=nodes, layers=layers,
                heads=heads, kv_heads=kv_heads, dim=dim, kv=kv, act=act, page=16)


def _handoff(name, seqs, lo, hi, layers, kv_heads, dim, kv):
    return dict(name=name, kind="handoff", seqs=seqs, lo=lo, hi=hi, layers=layers, kv_heads=kv_heads, dim=dim, kv=kv,
                act="fp32" if kv in ("fp32", "int8") else "fp16", page=16)


def draw(rng):
    def log_uniform(a, b):
        return max(a, min(b, int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))))

    kind = rng.choice(["step", "step", "step", "prompt", "verify", "handoff"])
    kv = rng.choice(["fp16", "int8blk", "int8blk", "fp32", "int8"])
    act = "fp32" if kv in ("fp32", "int8") else rng.choice(["fp16", "fp16", "fp32"])
    kv_heads = rng.choice([2, 4, 8, 8])
    dim = rng.choice([128, 128, 128, 64, 96])
    heads = kv_heads * rng.choice([1, 2, 4, 4, 7, 8])
    page = rng.choice([16, 16, 16, 32, 64])
    rope = rng.choice(["half", "interleaved"])
    row = kv_heads * dim * 2 * CODE_BYTES[kv]
    if kind == "step":
        seqs, hi = log_uniform(1, 64), log_uniform(64, 32768)
        hi = min(hi, max(64, 2_000_000_000 // (row * seqs)))
        lo = hi if rng.random() < 0.3 else max(1, int(hi * rng.uniform(0.1, 0.9)))
        c = _step("", seqs, lo, hi, heads, kv_heads, dim, kv, act, page, rng.choice([rope, "none"]))
    elif kind == "prompt":
        seqs, hi = log_uniform(1, 16), log_uniform(16, 4096)
        c = _prompt("", seqs, max(1, int(hi * rng.uniform(0.3, 1.0))), hi, heads, kv_heads, dim, kv, act, page, rope)
    elif kind == "verify":
        seqs, prefix = log_uniform(1, 128), 16 * rng.choice([0, 0, log_uniform(16, 256)])
        hi = log_uniform(64, 1024 if prefix else 4096)
        hi = min(hi, max(64, 400_000_000 // (row * seqs)))
        c = _verify("", seqs, prefix, max(0 if prefix else 1, int(hi * rng.uniform(0.0, 0.9))), hi, rng.randint(3, 24),
                    2, heads, kv_heads, dim, kv, act)
    else:
        seqs, hi = log_uniform(1, 8), log_uniform(64, 4096)
        c = _handoff("", seqs, max(1, int(hi * rng.uniform(0.3, 1.0))), hi, rng.choice([2, 4, 8]), kv_heads, dim, kv)
    del c["name"]
    return c


# ---- sizes -----------------------------------------------------------------------------------------

def _lengths(case):
    """The sequences' lengths (verify: past the shared prefix), the same for every seed."""
    r = np.random.Generator(np.random.PCG64(case["seqs"] * 1_000_003 + case["lo"] * 101 + case["hi"]))
    return r.integers(case["lo"], case["hi"] + 1, case["seqs"]).astype(np.int64)


def _pages(tokens, page):
    return -(-tokens // page)


def _act_bytes(case):
    return 4 if case["act"] == "fp32" else 2


def _kv_bytes(case, tokens):
    """Codes and scales of `tokens` cached tokens (an array of sequences' counts), K and V, one layer."""
    tokens = np.asarray(tokens)
    scales = {"int8blk": 2 * _pages(tokens, TILE), "int8": 4 * tokens}.get(case["kv"], 0 * tokens)
    return int(2 * case["kv_heads"] * (tokens * case["dim"] * CODE_BYTES[case["kv"]] + scales).sum())


def work(case):
    lens = _lengths(case)
    hq, hkv, dim, act = case.get("heads", 0), case["kv_heads"], case["dim"], _act_bytes(case)
    if case["kind"] == "step":
        s = case["seqs"]
        new = 2 * s * hkv * dim * (act + CODE_BYTES[case["kv"]])
        table = 4 * int(_pages(lens, case["page"]).sum())
        return {"bytes": _kv_bytes(case, lens) + new + table + s * hq * dim * (act + 4),
                "flops": 4.0 * hq * dim * float(lens.sum())}
    if case["kind"] == "prompt":
        t = int(lens.sum())
        return {"bytes": 2 * t * hkv * dim * act + _kv_bytes(case, lens) + 2 * t * hq * dim * act + 12 * t
                + 4 * dim * int(lens.max()), "flops": 0}
    if case["kind"] == "verify":
        s, n = case["seqs"], case["nodes"]
        ctx = lens + case["prefix"]
        draft = 2 * s * n * hkv * dim * (act + CODE_BYTES[case["kv"]])
        table = 4 * int(_pages(ctx + n, TILE).sum())
        layer = (_kv_bytes(case, [case["prefix"]]) + _kv_bytes(case, lens + n) + draft + table
                 + s * n * hq * dim * (act + 4))
        cow = 2 * _kv_bytes(case, np.full(int((ctx % TILE > 0).sum()), TILE))
        return {"bytes": case["layers"] * (layer + cow), "flops": 4.0 * case["layers"] * n * hq * dim * float((ctx + n).sum())}
    pages = TILE * _pages(lens, TILE)
    return {"bytes": 4 * case["layers"] * _kv_bytes(case, pages), "flops": 0}


def tolerance(case):
    if case["kind"] == "handoff":
        return "exact"
    if case["kind"] == "prompt":  # rotated rows: each value rounded once to its type
        return {"rel": 1e-3 if case["act"] == "fp16" else 5e-7}
    # attention: fp32 throughout over an fp32 cache; over the others probabilities and values meet in fp16
    return {"rel": 3e-6, "max": 5e-5} if case["kv"] == "fp32" else {"rel": 2e-3, "max": 0.1}


# ---- inputs ----------------------------------------------------------------------------------------

@functools.lru_cache(None)
def _context():
    return velokv.Context(0)


@functools.lru_cache(None)
def _rope_table(dim, n_pos):
    return torch.from_numpy(velokv.rope_table(n_pos, dim, ROPE_BASE)).cuda()


class _Rows:
    """Seeded K and V rows, N(0, 1); for the compressed caches 1 % of the channels are eight times larger."""

    def __init__(self, case, seed):
        self.case, self.gen = case, torch.Generator("cuda")
        self.gen.manual_seed(seed)
        self.dtype = torch.float32 if case["act"] == "fp32" else torch.float16
        shape = (case["kv_heads"], case["dim"])
        big = torch.rand(shape, generator=self.gen, device="cuda") < 0.01
        self.gain = torch.where(big, 8.0, 1.0).to(self.dtype) if case["kv"].startswith("int8") else None

    def kv(self, n):
        x = torch.randn((n, self.case["kv_heads"], self.case["dim"]), generator=self.gen, device="cuda", dtype=self.dtype)
        return x if self.gain is None else x.mul_(self.gain)

    def q(self, *lead):
        return torch.randn((*lead, self.case["heads"], self.case["dim"]), generator=self.gen, device="cuda", dtype=self.dtype)


class _Raw:
    """Device memory of a pool as a torch tensor reads it; keeps the pool."""

    def __init__(self, pool, ptr, count, kind):
        self.pool = pool
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": kind, "data": (ptr, False), "version": 2}


def _views(pool, case, floats=False):
    """The pool's contents, layer by layer: codes (as bytes or words; floats=True: as numbers) and scales."""
    kind = {"fp32": "<f4" if floats else "<i4", "fp16": "<f2" if floats else "<i2"}.get(case["kv"], "|i1")
    got = []
    for layer in range(pool.n_layer):
        v = pool.layer_view(layer)
        count = v.codes_bytes // CODE_BYTES[case["kv"]]
        parts = [(v.k_codes, count, kind), (v.v_codes, count, kind)]
        if case["kv"] == "int8blk":  # one word holds a block's K and V scale
            parts.append((v.k_scales, v.scales_bytes // 2, "<i4"))
        elif case["kv"] == "int8":
            parts += [(v.k_scales, v.scales_bytes // 4, "<i4"), (v.v_scales, v.scales_bytes // 4, "<i4")]
        got.append([torch.as_tensor(_Raw(pool, *p), device="cuda") for p in parts])
    return got


def _tables(n_pages, counts, seed):
    """Block tables: a random scatter of the pool's pages over the sequences."""
    perm = np.random.Generator(np.random.PCG64(seed)).permutation(n_pages).astype(np.int32)
    table = np.zeros((len(counts), int(max(counts))), np.int32)
    at = 0
    for s, n in enumerate(counts):
        table[s, :n] = perm[at:at + n]
        at += n
    return table


def _positions(lens):
    """(sequence, position) of every token of sequences of these lengths."""
    seq = torch.repeat_interleave(torch.arange(len(lens)), torch.from_numpy(lens)).cuda()
    first = torch.from_numpy(np.cumsum(lens) - lens).cuda()
    return seq, torch.arange(int(lens.sum()), device="cuda") - first[seq]


def _slots(table, seq, pos, page):
    return table[seq, torch.div(pos, page, rounding_mode="floor")].to(torch.int64) * page + pos % page


def _pool(case, n_pages, layers=1):
    return velokv.Pool(_context(), layers, n_pages, case["page"], case["kv_heads"], case["dim"], KV_TYPES[case["kv"]])


def _dt(case):
    return velokv.DT_F32 if case["act"] == "fp32" else velokv.DT_F16


def prepare(case, seed):
    return {"step": _prepare_step, "prompt": _prepare_prompt, "verify": _prepare_verify,
            "handoff": _prepare_handoff}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _step_rows(case, seed, lens):
    rows = _Rows(case, seed)
    past = int(lens.sum()) - len(lens)
    return rows.kv(past), rows.kv(past), rows.kv(len(lens)), rows.kv(len(lens)), rows.q(len(lens))


def _prepare_step(case, seed):
    ctx, lens, page = _context(), _lengths(case), case["page"]
    pages = _pages(lens, page)
    n_pages = int(pages.sum()) * 5 // 4 + 8
    table = torch.from_numpy(_tables(n_pages, pages, seed)).cuda()
    pool = _pool(case, n_pages)
    k, v, k_new, v_new, q = _step_rows(case, seed, lens)
    if k.shape[0]:
        seq, pos = _positions(lens - 1)
        slots = _slots(table, seq, pos, page)
        ctx.append(pool, 0, k.data_ptr(), v.data_ptr(), _dt(case), slots.data_ptr(), k.shape[0])
        torch.cuda.synchronize()
    del k, v
    out = torch.empty(q.shape, dtype=torch.float32, device="cuda")
    d_lens = torch.from_numpy(lens.astype(np.int32)).cuda()
    top = int(lens.max())
    call = dict(q=q.data_ptr(), q_dtype=_dt(case), out=out.data_ptr(), context_lens=d_lens.data_ptr(), n_seqs=len(lens),
                n_heads=case["heads"], max_context_len=top, block_tables=table.data_ptr(), bt_stride=table.shape[1],
                sum_context_len=int(lens.sum()), k_new=k_new.data_ptr(), v_new=v_new.data_ptr(), in_dtype=_dt(case))
    keep = [table, k_new, v_new, q, d_lens]
    if case["rope"] != "none":
        cs = _rope_table(case["dim"], -(-top // 1024) * 1024)
        call.update(cos_sin=cs.data_ptr(), n_pos=cs.shape[0], rope_style=STYLES[case["rope"]])
        keep.append(cs)
    return {"run": _run_step, "ctx": ctx, "pool": pool, "call": call, "rope": case["rope"] != "none", "keep": keep,
            "answer": [out, _views(pool, case)]}


def _run_step(st):
    one = st["ctx"].append_rope_decode if st["rope"] else st["ctx"].append_decode
    one(st["pool"], 0, **st["call"])
    return st["answer"]


def _prompt_rows(case, seed, lens):
    rows, t = _Rows(case, seed), int(lens.sum())
    return rows.kv(t), rows.kv(t), rows.q(t)


def _prepare_prompt(case, seed):
    ctx, lens, page = _context(), _lengths(case), case["page"]
    pages = _pages(lens, page)
    n_pages = int(pages.sum()) * 5 // 4 + 8
    table = torch.from_numpy(_tables(n_pages, pages, seed)).cuda()
    pool = _pool(case, n_pages)
    k, v, q = _prompt_rows(case, seed, lens)
    seq, pos = _positions(lens)
    slots, pos = _slots(table, seq, pos, page), pos.to(torch.int32)
    cs = _rope_table(case["dim"], -(-int(lens.max()) // 1024) * 1024)
    call = dict(k=k.data_ptr(), v=v.data_ptr(), in_dtype=_dt(case), positions=pos.data_ptr(), slot_mapping=slots.data_ptr(),
                n_tok=k.shape[0], cos_sin=cs.data_ptr(), n_pos=cs.shape[0], style=STYLES[case["rope"]], q=q.data_ptr(),
                q_dtype=_dt(case), n_heads=case["heads"])
    return {"run": _run_prompt, "ctx": ctx, "pool": pool, "call": call, "keep": [k, v, pos, slots, cs],
            "answer": [q, _views(pool, case, floats=True)]}


def _run_prompt(st):
    st["ctx"].append_rope(st["pool"], 0, **st["call"])
    return st["answer"]


def _verify_plan(case, seed):
    """Tables, the copy-on-write pairs, the tree and the accepted paths of a speculative step."""
    n, lens, prefix = case["nodes"], _lengths(case), case["prefix"]
    r = np.random.Generator(np.random.PCG64(seed))
    ctx = lens + prefix
    shared = prefix // TILE
    own = _pages(ctx + n, TILE) - shared
    partial = lens % TILE > 0
    n_pages = (shared + int(own.sum()) + int(partial.sum())) * 9 // 8 + 8
    perm = r.permutation(n_pages).astype(np.int32)
    table = np.zeros((len(lens), shared + int(own.max())), np.int32)
    table[:, :shared] = perm[:shared]
    at = shared
    for s, p in enumerate(own):
        table[s, shared:shared + p] = perm[at:at + p]
        at += p
    filled, pairs = table.copy(), []
    for s in np.nonzero(partial)[0]:  # the partial block as the cache holds it, and the sequence's own copy
        col = int(ctx[s]) // TILE
        filled[s, col] = perm[at]
        pairs.append((int(perm[at]), int(table[s, col])))
        at += 1
    tree = velokv.branching_tree([2] * 8, n)
    accept, count = np.full((len(lens), 32), -1, np.int32), np.zeros(len(lens), np.int32)
    for s in range(len(lens)):
        path = tree.path_nodes(int(r.integers(0, n)))
        accept[s, :len(path)], count[s] = path, len(path)
    return lens, ctx, n_pages, table, filled, pairs, tree.ancestor_mask(), accept, count


def _verify_rows(case, seed, lens):
    """Per layer: K and V of the prefix and the suffixes, then of the drafts, and q."""
    rows, s, n = _Rows(case, seed), case["seqs"], case["nodes"]
    past = case["prefix"] + int(lens.sum())
    for _ in range(case["layers"]):
        yield rows.kv(past), rows.kv(past), rows.kv(s * n), rows.kv(s * n), rows.q(s, n)


def _prepare_verify(case, seed):
    ctx, s, n = _context(), case["seqs"], case["nodes"]
    lens, total, n_pages, table, filled, pairs, mask, accept, count = _verify_plan(case, seed)
    pool = _pool(case, n_pages, case["layers"])
    d_table, d_filled = torch.from_numpy(table).cuda(), torch.from_numpy(filled).cuda()
    seq, pos = _positions(lens)
    head = torch.arange(case["prefix"], device="cuda")
    fill = torch.cat([_slots(d_filled, torch.zeros_like(head), head, TILE), _slots(d_filled, seq, pos + case["prefix"], TILE)])
    d_total = torch.from_numpy(total).cuda()
    at = (d_total[:, None] + torch.arange(n, device="cuda")[None, :]).reshape(-1)
    drafts = _slots(d_table, torch.arange(s, device="cuda").repeat_interleave(n), at, TILE)
    layers = []
    for layer, (k, v, dk, dv, q) in enumerate(_verify_rows(case, seed, lens)):
        if k.shape[0]:
            ctx.append(pool, layer, k.data_ptr(), v.data_ptr(), _dt(case), fill.data_ptr(), k.shape[0])
        layers.append((dk, dv, q, torch.empty(q.shape, dtype=torch.float32, device="cuda")))
        torch.cuda.synchronize()
    d_total = d_total.to(torch.int32)
    d_mask = torch.from_numpy(np.tile(mask, s).astype(np.int32)).cuda()
    d_accept, d_count = torch.from_numpy(accept).cuda(), torch.from_numpy(count).cuda()
    status = torch.zeros(s, dtype=torch.int32, device="cuda")
    table_at = dict(block_tables=d_table.data_ptr(), bt_stride=table.shape[1])
    verify = dict(q_dtype=_dt(case), context_lens=d_total.data_ptr(), tree_mask=d_mask.data_ptr(), n_seqs=s, n_nodes=n,
                  n_heads=case["heads"], max_context_len=int(total.max()), shared_blocks=case["prefix"] // TILE, **table_at)
    commit = dict(context_lens=d_total.data_ptr(), accept=d_accept.data_ptr(), accept_stride=32, n_accept=d_count.data_ptr(),
                  n_seqs=s, status=status.data_ptr(), **table_at)
    return {"run": _run_verify, "ctx": ctx, "pool": pool, "pairs": np.array(pairs, np.int32).reshape(-1, 2), "dt": _dt(case),
            "drafts": drafts, "n_draft": s * n,
            "layers": [(dk.data_ptr(), dv.data_ptr(), q.data_ptr(), out.data_ptr()) for dk, dv, q, out in layers],
            "verify": verify, "commit": commit, "keep": [layers, d_table, d_total, d_mask, d_accept, d_count],
            "answer": [[out for *_, out in layers], status, _views(pool, case)]}


def _run_verify(st):
    ctx, pool = st["ctx"], st["pool"]
    if len(st["pairs"]):
        ctx.copy_blocks(pool, st["pairs"])
    slots = st["drafts"].data_ptr()
    for layer, (dk, dv, q, out) in enumerate(st["layers"]):
        ctx.append(pool, layer, dk, dv, st["dt"], slots, st["n_draft"])
        ctx.tree_verify(pool, layer, q, out=out, **st["verify"])
    ctx.tree_commit(pool, **st["commit"])
    return st["answer"]


def _prepare_handoff(case, seed):
    ctx, lens, nl = _context(), _lengths(case), case["layers"]
    pages = _pages(lens, TILE)
    used = int(pages.sum())
    n_pages = used * 5 // 4 + 8
    src, dst = _pool(case, n_pages, nl), _pool(case, n_pages, nl)
    table = _tables(n_pages, pages, seed)
    d_table = torch.from_numpy(table).cuda()
    rows = _Rows(case, seed)
    seq, pos = _positions(lens)
    slots = _slots(d_table, seq, pos, TILE)
    for layer in range(nl):
        k, v = rows.kv(len(seq)), rows.kv(len(seq))
        ctx.append(src, layer, k.data_ptr(), v.data_ptr(), _dt(case), slots.data_ptr(), len(seq))
        torch.cuda.synchronize()
    items, first, offset = [], 0, 0
    for s, n in enumerate(lens):
        items.append((1000 + s, int(n), first, offset))
        first += int(pages[s])
        offset += -(-(velokv.NIXL_HEADER_BYTES + src.nixl_payload_bytes(int(n))) // 16) * 16
    flat = np.concatenate([table[s, :n] for s, n in enumerate(pages)])
    here = torch.from_numpy(flat).cuda()
    there = torch.from_numpy(np.random.Generator(np.random.PCG64(seed + 1)).permutation(n_pages)[:used].astype(np.int32)).cuda()
    wire = torch.zeros(offset, dtype=torch.uint8, device="cuda")
    packed = torch.full((len(items),), -1, dtype=torch.int32, device="cuda")
    unpacked = packed.clone()
    return {"run": _run_handoff, "ctx": ctx, "src": src, "dst": dst, "items": items, "used": used, "here": here, "there": there,
            "wire": wire, "packed": packed, "unpacked": unpacked, "answer": [wire, packed, unpacked, _views(dst, case)]}


def _run_handoff(st):
    ctx, wire, size = st["ctx"], st["wire"].data_ptr(), st["wire"].numel()
    ctx.nixl_pack(st["src"], st["items"], st["here"].data_ptr(), st["used"], wire, size, st["packed"].data_ptr())
    ctx.nixl_unpack(st["dst"], st["items"], st["there"].data_ptr(), st["used"], wire, size, st["unpacked"].data_ptr())
    return st["answer"]


# ---- the same in 64 bits ---------------------------------------------------------------------------

def _rotate(x, pos, style):
    """x [tokens, heads, dim] in 64 bits, rotated at its tokens' positions."""
    dim = x.shape[-1]
    angle = pos.double()[:, None] * ROPE_BASE ** (-2.0 * torch.arange(dim // 2, device=x.device, dtype=torch.float64) / dim)
    c, s = angle.cos()[:, None, :], angle.sin()[:, None, :]
    y = torch.empty_like(x)
    a, b = (slice(0, dim, 2), slice(1, dim, 2)) if style == "interleaved" else (slice(0, dim // 2), slice(dim // 2, dim))
    y[..., a], y[..., b] = x[..., a] * c - x[..., b] * s, x[..., a] * s + x[..., b] * c
    return y


def _cached(x, kv):
    """The values a cache of this type holds for the rows x [tokens, heads, dim], appended in order from a block's first slot."""
    if kv == "fp32":
        return x.float().double()
    if kv == "fp16":
        return x.half().double()
    x, top = x.float(), torch.full((1,), 127.0, device=x.device)  # a tensor: torch divides by a number with its reciprocal
    if kv == "int8":  # per token and head: scale amax / 127, codes truncated
        amax = x.abs().amax(-1, keepdim=True)
        code = torch.where(amax > 0, x * (top / amax), 0.0).trunc()
        return code.double() * (amax / top).double()
    n = x.shape[0]
    x = torch.nn.functional.pad(x, (0, 0, 0, 0, 0, -n % TILE)).view(-1, TILE, *x.shape[1:])
    code, scale = torch.zeros_like(x), torch.zeros_like(x[:, 0, :, :1])
    for t in range(TILE):  # the block's scale grows with its tokens, the codes before follow
        new = torch.maximum(scale, (x[:, t].abs().amax(-1, keepdim=True) / top).half().float())
        grown = torch.where(new > 0, new, 1.0)
        code[:, :t] = torch.where((new > scale)[:, None], (code[:, :t] * scale[:, None] / grown[:, None]).round().clamp(-127, 127), code[:, :t])
        code[:, t] = torch.where(new > 0, (x[:, t] / grown).round().clamp(-127, 127), 0.0)
        scale = new
    return (code.double() * scale[:, None].double()).view(-1, *x.shape[2:])[:n]


def _attend(q, k, v, mask=None):
    """q [rows, heads, dim] over k, v [tokens, kv_heads, dim]; mask [rows, tokens]: the tokens a row sees."""
    rows, heads, dim = q.shape
    group = heads // k.shape[1]
    qq = q.double().view(rows, -1, group, dim).permute(1, 0, 2, 3).reshape(k.shape[1], rows * group, dim)
    score = qq @ k.permute(1, 2, 0).contiguous() / math.sqrt(dim)
    if mask is not None:
        score = score.masked_fill(~mask[None].repeat_interleave(group, 1), -math.inf)
    o = torch.softmax(score, -1) @ v.permute(1, 0, 2).contiguous()
    return o.view(-1, rows, group, dim).permute(1, 0, 2, 3).reshape(rows, heads, dim)


def _no_views(case, layers=1):
    return [[None] * {"int8blk": 3, "int8": 4}.get(case["kv"], 2) for _ in range(layers)]


def _float_pool(case, rows, slots, n_pages, is_v):
    """A pool layer's K or V codes of a float cache after these rows: tiles of 16 tokens, token pairs interleaved for V."""
    dim, width = case["dim"], 64 if case["dim"] <= 64 else 128
    x = torch.zeros((n_pages * case["page"], case["kv_heads"], width), dtype=torch.float64, device="cuda")
    x[slots, :, :dim] = _cached(rows, case["kv"])
    x = x.view(-1, TILE, case["kv_heads"], width).transpose(1, 2)
    if is_v:
        x = x.reshape(x.shape[0], x.shape[1], TILE // 2, 2, width).transpose(3, 4)
    return x.reshape(-1)


def exact(case, seed):
    lens = _lengths(case)
    if case["kind"] == "handoff":
        return None
    if case["kind"] == "step":
        k, v, k_new, v_new, q = _step_rows(case, seed, lens)
        at = torch.from_numpy(lens - 1).cuda()
        k_new, q = k_new.double(), q.double()
        if case["rope"] != "none":
            k_new, q = _rotate(k_new, at, case["rope"]), _rotate(q, at, case["rope"])
        out, first = [], 0
        for s, n in enumerate(lens):
            past = slice(first, first + int(n) - 1)
            first += int(n) - 1
            kk = _cached(torch.cat([k[past].double(), k_new[s:s + 1]]), case["kv"])
            vv = _cached(torch.cat([v[past], v_new[s:s + 1]]), case["kv"])
            out.append(_attend(q[s:s + 1], kk, vv))
        return [torch.cat(out), _no_views(case)]
    if case["kind"] == "prompt":
        k, v, q = _prompt_rows(case, seed, lens)
        seq, pos = _positions(lens)
        q, k = _rotate(q.double(), pos, case["rope"]), _rotate(k.double(), pos, case["rope"])
        if case["kv"].startswith("int8"):
            return [q, _no_views(case)]
        pages = _pages(lens, case["page"])
        n_pages = int(pages.sum()) * 5 // 4 + 8
        slots = _slots(torch.from_numpy(_tables(n_pages, pages, seed)).cuda(), seq, pos, case["page"])
        return [q, [[_float_pool(case, k, slots, n_pages, False), _float_pool(case, v.double(), slots, n_pages, True)]]]
    n, prefix = case["nodes"], case["prefix"]
    mask = torch.from_numpy(_verify_plan(case, seed)[6].astype(np.int64)).cuda()
    sees = (mask[:, None] >> torch.arange(n, device="cuda")[None, :] & 1).bool()
    outs = []
    for k, v, dk, dv, q in _verify_rows(case, seed, lens):
        out, first = [], prefix
        heads = [_cached(x[:prefix], case["kv"]) for x in (k, v)]
        for s, m in enumerate(lens):
            own, draft = slice(first, first + int(m)), slice(s * n, (s + 1) * n)
            first += int(m)
            kk, vv = (torch.cat([h, _cached(torch.cat([x[own], d[draft]]), case["kv"])]) for h, x, d in zip(heads, (k, v), (dk, dv)))
            past = torch.ones((n, prefix + int(m)), dtype=torch.bool, device="cuda")
            out.append(_attend(q[s], kk, vv, torch.cat([past, sees], 1)))
        outs.append(torch.stack(out))
    return [outs, None, _no_views(case, case["layers"])]
