"""KVQ_DEBUG_DUMP: the long-query path's attention call, saved for an offline replay.

The reference saves the metadata of its last FlashAttention call (kvq/cuda_kernels.py:123-127) and
replays it with random tensors of the same shapes (scripts/replay_fa_call.py) -- the tool that located
its mixed-batch memory fault (docs/WALKTHROUGH.md:357-370). Here the long path's consumer is a HIP
prefill kernel, so a dump holds what that call reads: the query start offsets and the device key counts,
the work list as it runs (pieces, slots and merge list of cut rows included), which source it reads -- the
temporary cache, with its block table and page sources, or the INT8 pages through the requests' own table --
and the shapes and strides of q, out and both caches.

    dump_long_call(path, ...)   called by cuda_kernels.long_attention while KVQ_DEBUG_DUMP=path
    load(path)                  the dump (torch.load with weights_only=True: tensors and plain values)
    check(d)                    host-side bounds report of a dump: the reads and writes the call would make
    replay(d, seed)             the same call on random tensors of the dumped shapes, on the GPU

Dumps without a work list's pieces or the INT8 cache (older files) are checked and replayed as whole rows of
the temporary cache.
"""
import torch

FIELDS = ("cu_seqlens_q", "seq_lens", "block_table", "src_req", "src_j", "tile_req", "tile_row")
SPLIT_FIELDS = ("tile_piece", "tile_slot", "merge")
MAX_PARTS = 64         # pieces an entry's keys may be cut into (kvq_prefill_max_parts)
REPLAY_SCALE = 1 / 64  # every K and V scale of a replayed direct call


def dump_long_call(path, q, out, cu_seqlens_q, seq_lens, plan, kt, tile_req, tile_row, max_query_len, rows_per_tile,
                   softmax_scale, work=None, source="0", caches=None):
    """Save the prefill call of one long_attention step (synchronises the device: a debugging aid). kt: the
    temporary cache or its shape. work: the call's cuda_kernels.PrefillWork, whose list stands in for tile_req /
    tile_row; source: "0" the temporary cache, "1" / "fold" the INT8 pages (KVQ_PREFILL_DIRECT's values); caches:
    (k_cache, v_cache, block_table, k_scale, v_scale) of the call."""
    src_req, src_j, bt = (torch.as_tensor(x) for x in (plan.src_req, plan.src_j, plan.block_table))
    if work is not None:
        tile_req, tile_row = work.tile_req, work.tile_row
    n = cu_seqlens_q.shape[0] - 1
    d = {"cu_seqlens_q": cu_seqlens_q.cpu(), "seq_lens": seq_lens.cpu()[:n].clone(),
         "block_table": bt.cpu(), "src_req": src_req.cpu(), "src_j": src_j.cpu(), "tile_req": tile_req.cpu(),
         "tile_row": tile_row.cpu(), "max_seqlen_q": int(max_query_len), "max_seqlen_k": int(plan.max_seqlen_k),
         "q_shape": tuple(q.shape), "q_stride": tuple(q.stride()), "out_shape": tuple(out.shape),
         "out_stride": tuple(out.stride()), "kt_shape": tuple(getattr(kt, "shape", kt)), "block_size": int(plan.block_size),
         "rows_per_tile": int(rows_per_tile), "softmax_scale": float(softmax_scale), "source": source}
    if work is not None and work.tile_piece is not None:
        d.update(tile_piece=work.tile_piece.cpu(), tile_slot=work.tile_slot.cpu(), merge=work.merge.cpu(),
                 slots=int(work.slots))
    if caches is not None:
        kc, vc, table, ks, vs = caches
        one = kc.untyped_storage().data_ptr() == vc.untyped_storage().data_ptr()
        d.update(cache_table=table[:n].cpu(), cache_shape=tuple(kc.shape), k_stride=tuple(kc.stride()),
                 v_stride=tuple(vc.stride()), scale_cols=(int(ks.shape[-1]), int(vs.shape[-1])),
                 v_offset=vc.storage_offset() - kc.storage_offset() if one else None)   # None: caches of their own
    torch.save(d, path)
    return d


def load(path):
    return torch.load(path, weights_only=True)


def check(d):
    """Every read the prefill call would make, and every write of its pieces, checked on the host: a list of
    problems (empty if none). For each work-list entry (request r, first row r0): its rows lie in r's query rows;
    r's key count is at least its query count; the keys it reads, [0, seq_lens[r]), lie on pages of r's row of the
    table the call reads -- the temporary cache's, whose entries are pages copied from request r, in order, or the
    requests' own, whose entries are pages of the INT8 cache. The copies read pages of that cache too. Rows cut
    into pieces: every piece once, in its merge entry's slot, inside the partial buffers; every cut row merged
    once."""
    errs = []
    cu, sl, bt = d["cu_seqlens_q"].long(), d["seq_lens"].long(), d["block_table"].long()
    src_req, src_j = d["src_req"].long(), d["src_j"].long()
    T, hq, _ = d["q_shape"]
    P, bs, hkv, _ = d["kt_shape"]
    G = hq // hkv
    n = cu.numel() - 1
    ql = cu[1:] - cu[:-1]
    direct = d.get("source", "0") != "0"
    table = d["cache_table"].long() if "cache_table" in d else None
    if int(cu[-1]) > T:
        errs.append(f"cu_seqlens_q[-1] {int(cu[-1])} > {T} query rows")
    if src_req.numel() != P or src_j.numel() != P:
        errs.append(f"{src_req.numel()} page sources for {P} temporary pages")
    if table is not None and not direct:
        for r, j in zip(src_req.tolist(), src_j.tolist()):
            if not (0 <= r < n and 0 <= j < table.shape[1]):
                errs.append(f"req {r}: page {j} to copy outside the block table")
            elif not 0 <= int(table[r, j]) < d["cache_shape"][0]:
                errs.append(f"req {r}: page {j} to copy is id {int(table[r, j])} of {d['cache_shape'][0]}")
    for r, r0 in sorted(set(zip(d["tile_req"].long().tolist(), d["tile_row"].long().tolist()))):
        if not 0 <= r < n:
            errs.append(f"work entry for request {r} of {n}")
            continue
        if not 0 <= r0 < int(ql[r]) * G:
            errs.append(f"req {r}: work rows from {r0}, request has {int(ql[r]) * G} rows")
        L = int(sl[r])
        if L < int(ql[r]):
            errs.append(f"req {r}: {L} keys < {int(ql[r])} query tokens")
        pages = -(-L // bs)
        reads, count, what = (table, d["cache_shape"][0], "page ids") if direct else (bt, P, "temporary page ids")
        if pages > reads.shape[1]:
            errs.append(f"req {r}: {pages} pages > block table width {reads.shape[1]}")
            continue
        ids = reads[r, :pages]
        if pages and (int(ids.min()) < 0 or int(ids.max()) >= count):
            errs.append(f"req {r}: {what} outside [0, {count})")
            continue
        if not direct and pages and not (bool((src_req[ids] == r).all()) and torch.equal(src_j[ids], torch.arange(pages))):
            errs.append(f"req {r}: its table row points at pages copied from other requests or out of order")
    return errs + (_check_pieces(d) if "tile_piece" in d else [])


def _check_pieces(d):
    errs, rows = [], {}
    for r, r0, p, slot in zip(*(d[k].long().tolist() for k in ("tile_req", "tile_row", "tile_piece", "tile_slot"))):
        part, parts = p & 0xffff, p >> 16
        if not 0 <= part < parts <= MAX_PARTS:
            errs.append(f"req {r}: rows from {r0}, piece {part} of {parts}")
        rows.setdefault((r, r0), []).append((part, parts, slot))
    merge = {}
    for r, r0, first, parts in d["merge"].long().tolist():
        if (r, r0) in merge:
            errs.append(f"req {r}: rows from {r0} merged twice")
        merge[r, r0] = first, parts
        if not (0 <= first and first + parts <= d["slots"]):
            errs.append(f"req {r}: rows from {r0}, slots {first} .. {first + parts - 1} of {d['slots']} merged")
    used = {}
    for (r, r0), pieces in rows.items():
        n = pieces[0][1]
        if sorted(p for p, _, _ in pieces) != list(range(n)) or any(m != n for _, m, _ in pieces):
            errs.append(f"req {r}: rows from {r0}, pieces {sorted(p for p, _, _ in pieces)} of {n}")
        first, merged = merge.pop((r, r0), (None, 1))
        if merged != n:
            errs.append(f"req {r}: rows from {r0}, {n} pieces, {merged} merged")
        for part, _, slot in pieces if n > 1 else ():
            if not 0 <= slot < d["slots"]:
                errs.append(f"req {r}: rows from {r0}, slot {slot} of {d['slots']}")
            elif used.setdefault(slot, (r, r0, part)) != (r, r0, part):
                errs.append(f"req {r}: rows from {r0}, slot {slot} also written by req {used[slot][0]}")
            if first is not None and slot != first + part:
                errs.append(f"req {r}: rows from {r0}, piece {part} in slot {slot}, merged from {first + part}")
    return errs + [f"req {r}: rows from {r0} merged but not in the work list" for r, r0 in merge]


def _random_caches(d, g, device):
    """INT8 K and V caches of the dumped shape and strides, in one storage where they were."""
    shape, sizes = d["cache_shape"], []
    for stride, offset in ((d["k_stride"], 0), (d["v_stride"], d["v_offset"] or 0)):
        sizes.append(offset + 1 + sum((s - 1) * st for s, st in zip(shape, stride)))
    if d["v_offset"] is None:
        stores = [torch.empty(n, dtype=torch.int8, device=device) for n in sizes]
        k, v = stores[0].as_strided(shape, d["k_stride"]), stores[1].as_strided(shape, d["v_stride"])
    else:
        at = max(0, -d["v_offset"])
        stores = [torch.empty(at + max(sizes), dtype=torch.int8, device=device)]
        k = stores[0].as_strided(shape, d["k_stride"], at)
        v = stores[0].as_strided(shape, d["v_stride"], at + d["v_offset"])
    for s in stores:
        s.random_(-127, 128, generator=g)
    return k, v


def replay(d, seed=0, device="cuda"):
    """Run the dumped prefill call on random tensors of the dumped shapes and strides, on the GPU: q and the
    temporary K and V, or q and INT8 caches with every scale REPLAY_SCALE for a call that read the pages itself.
    Returns (q, kt, vt, out): the temporary K and V, for a direct call what they would be, and out, which holds the
    rows the work list covers, NaN elsewhere."""
    from . import cuda_kernels as ck

    g = torch.Generator(device=device).manual_seed(seed)
    T, hq, D = d["q_shape"]
    qs, os_ = d["q_stride"], d["out_stride"]
    q = torch.randn(T * qs[0], generator=g, device=device).to(torch.bfloat16).as_strided((T, hq, D), qs)
    out = torch.full((T * os_[0],), float("nan"), dtype=torch.bfloat16, device=device).as_strided((T, hq, D), os_)
    idx = {k: d[k].to(device=device, dtype=torch.int32) for k in FIELDS + SPLIT_FIELDS + ("cache_table",) if k in d}
    split = None
    if "tile_piece" in d:
        hkv, rows = d["kt_shape"][2], d["rows_per_tile"]
        split = (*(idx[k] for k in SPLIT_FIELDS),
                 *(torch.empty(d["slots"], hkv, rows, n, dtype=torch.float32, device=device) for n in (D, 2)))
    lists = idx["tile_req"], idx["tile_row"], d["softmax_scale"]
    if d.get("source", "0") != "0":
        k, v = _random_caches(d, g, device)
        scales = [torch.full((k.shape[2], n), REPLAY_SCALE, device=device) for n in d["scale_cols"]]
        ck.ext().int8_prefill_attention(q, k, v, out, idx["cu_seqlens_q"], idx["seq_lens"], idx["cache_table"], *lists, *scales,
                                        d["source"] == "fold", split)
        ids = d["cache_table"].long()[d["src_req"].long(), d["src_j"].long()]
        ids = torch.where((ids >= 0) & (ids < k.shape[0]), ids, 0).to(device)      # (as the kernels read them)
        return q, (k[ids] * REPLAY_SCALE).to(torch.bfloat16), (v[ids] * REPLAY_SCALE).to(torch.bfloat16), out
    kt = torch.randn(d["kt_shape"], generator=g, device=device).to(torch.bfloat16)
    vt = torch.randn(d["kt_shape"], generator=g, device=device).to(torch.bfloat16)
    ck.ext().paged_prefill_attention(q, kt, vt, out, idx["cu_seqlens_q"], idx["seq_lens"], idx["block_table"], *lists, split)
    return q, kt, vt, out
