"""KVQ_DEBUG_DUMP (kvq.debug_dump): the long path's prefill call saved for an offline replay, as the
reference's dump of its FlashAttention call (kvq/cuda_kernels.py:123-127) and scripts/replay_fa_call.py.

On the CPU: a dump of a mixed batch's call loads without unpickling code, its host-side bounds report is
clean, and replaying it through the oracle -- fp32 attention over the temporary cache its block table
describes, filled by the oracle's page dequantization -- reproduces implementation A on the original INT8
cache for every row the work list covers. Corrupted dumps (a table entry past the temporary cache, a key
count past the copied pages, a work entry past a request's rows, pages of another request) are reported.
On the GPU: the dump written by a real paged_attention call, replayed on the HIP prefill kernel, against
the oracle on the replay's tensors. Both with rows whole and cut into pieces, from the temporary cache and from the
INT8 pages.
"""
import os

import pytest
import torch
from conftest import record

from oracle import kvq_oracle as O
from kvq import cuda_kernels as ck
from kvq import debug_dump
from kvq import synth

ROWS = 128   # (token, q head) rows per work-list entry of the prefill kernel


def _batch(hq=28, hkv=4, d=128):
    q_lens, seq_lens = [1, 40, 3, 200, 1, 77], [100, 90, 300, 900, 17, 1500]
    c = synth.paged_case(hq, hkv, q_lens, seq_lens, head_dim=d, seed=91, dist="randn", scale=3.0)
    c["static"] = synth.scales_from(c["k"].reshape(-1, hkv, d), c["v"].reshape(-1, hkv, d))
    c["scale"] = d ** -0.5
    kq = O.quantize(c["k"].float() - c["static"]["k_mu"], c["static"]["k_scale"])
    vq = O.quantize(c["v"], c["static"]["v_scale"])
    return c, kq, vq


def oracle_replay(d, q, kt, vt):
    """The dumped call under the oracle: fp32 attention (paged_attention_ref) over the temporary cache for
    the requests the work list names; [T, Hq, D] with NaN on the other rows."""
    cu, sl, bt = d["cu_seqlens_q"], d["seq_lens"], d["block_table"]
    out = torch.full(q.shape, float("nan"))
    for r in sorted(set(d["tile_req"].tolist())):
        t0, t1 = int(cu[r]), int(cu[r + 1])
        cu_r = torch.tensor([0, t1 - t0], dtype=torch.int32)
        out[t0:t1] = O.paged_attention_ref(q[t0:t1].cpu().float(), kt.cpu(), vt.cpu(), cu_r, sl[r:r + 1], bt[r:r + 1],
                                           d["softmax_scale"]).float()
    return out


def _dump(tmp_path, c, kq, vq):
    plan = ck.plan_long(c["cu"], c["seq_lens"], 16)
    hq, hkv = c["q"].shape[1], c["k"].shape[2]
    tile_req, tile_row = plan.tiles(hq // hkv, "cpu", rows=ROWS)
    kt, vt = O.dequant_pages_ref(kq, vq, c["block_table"], torch.from_numpy(plan.src_req), torch.from_numpy(plan.src_j),
                                 c["static"])
    out = torch.empty_like(c["q"])
    path = str(tmp_path / "long_call.pt")
    debug_dump.dump_long_call(path, c["q"], out, c["cu"], c["seq_lens"], plan, kt, tile_req, tile_row,
                              int((c["cu"][1:] - c["cu"][:-1]).max()), ROWS, c["scale"])
    return path, plan, kt, vt


def test_dump_replays_through_the_oracle(tmp_path):
    c, kq, vq = _batch()
    path, plan, kt, vt = _dump(tmp_path, c, kq, vq)
    d = debug_dump.load(path)
    assert debug_dump.check(d) == []
    assert d["q_shape"] == tuple(c["q"].shape) and d["kt_shape"] == tuple(kt.shape)
    assert d["max_seqlen_k"] == 1500 and d["block_size"] == 16
    rep = oracle_replay(d, c["q"], kt, vt)
    ref = O.paged_static_attention(O.CFG32_Q32, c["static"], True, ck.SHORT_Q)(
        c["q"].float(), kq, vq, c["cu"], c["seq_lens"], c["block_table"], c["scale"])
    rows = torch.cat([torch.arange(int(c["cu"][r]), int(c["cu"][r + 1])) for r in plan.long_req.tolist()])
    e = O.compare(ref[rows], rep[rows])
    record("debug_dump_oracle_replay", **e)
    assert e["rel_l2"] < 1e-5, e
    covered = torch.zeros(c["q"].shape[0], dtype=torch.bool)
    covered[rows] = True
    assert torch.isnan(rep[~covered]).all() and not torch.isnan(rep[covered]).any()


@pytest.mark.parametrize("fault", ["page_past_cache", "keys_past_pages", "rows_past_request", "foreign_page"])
def test_check_reports_corrupted_dumps(tmp_path, fault):
    c, kq, vq = _batch()
    path, plan, kt, vt = _dump(tmp_path, c, kq, vq)
    d = debug_dump.load(path)
    r = int(plan.long_req[0])
    if fault == "page_past_cache":
        d["block_table"][r, 0] = kt.shape[0]
    elif fault == "keys_past_pages":
        d["seq_lens"][r] = 16 * d["block_table"].shape[1] + 1
    elif fault == "rows_past_request":
        i = int((d["tile_req"] == r).nonzero()[0])
        d["tile_row"][i] = 10 ** 6
    else:
        other = int(plan.long_req[1])
        d["block_table"][r, 0] = d["block_table"][other, 0]
    errs = debug_dump.check(d)
    assert errs and all(f"req {r}" in e for e in errs), errs


def _cut(monkeypatch, on=True):
    """Cut every row that can be (or none), whatever it is estimated to cost."""
    monkeypatch.setattr(ck, "_prefill_us", lambda longest, groups, partials, *a: (partials is None) == on)


def _dump_call(tmp_path, monkeypatch, source):
    """The dump of a long_attention call whose rows are cut, with the kernels left out."""
    class Nothing:
        calls, prefill_rows, prefill_max_parts = None, ROWS, 64

        def __getattr__(self, name):
            return lambda *a: None

    c, kq, vq = _batch()
    path = str(tmp_path / "cut.pt")
    monkeypatch.setattr(ck, "_EXT", Nothing())
    monkeypatch.setenv("KVQ_DEBUG_DUMP", path)
    monkeypatch.setenv("KVQ_PREFILL_DIRECT", source)
    _cut(monkeypatch)
    plan = ck.plan_long(c["cu"], c["seq_lens"], 16)
    ck.long_attention(c["q"], kq, vq, torch.empty_like(c["q"]), c["cu"], c["seq_lens"], c["block_table"], 200, plan,
                      c["scale"], c["static"])
    return debug_dump.load(path), plan.work(7, 4, 128, torch.device("cpu"))


@pytest.mark.parametrize("source", ["0", "1", "fold"])
def test_dump_holds_the_list_that_runs(tmp_path, monkeypatch, source):
    d, work = _dump_call(tmp_path, monkeypatch, source)
    assert debug_dump.check(d) == [] and d["source"] == source and d["slots"] == work.slots > 0
    for k in ("tile_req", "tile_row", "tile_piece", "tile_slot", "merge"):
        assert torch.equal(d[k], getattr(work, k)), k


@pytest.mark.parametrize("fault", ["slot_past_buffers", "slot_twice", "piece_of_none", "piece_missing", "merged_short",
                                   "merged_twice", "not_merged", "foreign_merge", "too_many_pieces"])
def test_check_reports_bad_pieces(tmp_path, monkeypatch, fault):
    d, _ = _dump_call(tmp_path, monkeypatch, "0")
    parts = d["tile_piece"] >> 16
    i = int((parts > 2).nonzero()[0])
    r, r0 = int(d["tile_req"][i]), int(d["tile_row"][i])
    m = int(((d["merge"][:, 0] == r) & (d["merge"][:, 1] == r0)).nonzero()[0])
    other = int((d["tile_slot"] != d["tile_slot"][i]).logical_and(parts > 1).nonzero()[0])
    if fault == "slot_past_buffers":
        d["tile_slot"][i] = d["slots"]
    elif fault == "slot_twice":
        d["tile_slot"][i] = d["tile_slot"][other]
    elif fault == "piece_of_none":
        d["tile_piece"][i] = int(parts[i]) << 16 | int(parts[i])
    elif fault == "piece_missing":
        for k in ("tile_req", "tile_row", "tile_piece", "tile_slot"):
            d[k] = torch.cat([d[k][:i], d[k][i + 1:]])
    elif fault == "merged_short":
        d["merge"][m, 3] -= 1
    elif fault == "merged_twice":
        d["merge"] = torch.cat([d["merge"], d["merge"][m:m + 1]])
    elif fault == "not_merged":
        d["merge"] = torch.cat([d["merge"][:m], d["merge"][m + 1:]])
    elif fault == "foreign_merge":
        d["merge"][m, 1] += ROWS * 1000
    else:
        same = (d["tile_req"] == r) & (d["tile_row"] == r0)
        d["tile_piece"][same] = (d["tile_piece"][same] & 0xffff) | 65 << 16
    errs = debug_dump.check(d)
    assert errs and any(f"req {r}" in e for e in errs), errs


@pytest.mark.parametrize("source", ["0", "1"])
@pytest.mark.parametrize("page", [-1, 10 ** 6])
def test_check_reports_pages_outside_the_int8_cache(tmp_path, monkeypatch, source, page):
    """Both sources start from the requests' own table: the direct kernel's pages, and the pages copied."""
    d, _ = _dump_call(tmp_path, monkeypatch, source)
    d["cache_table"][3, 5] = page
    errs = debug_dump.check(d)
    assert errs and all("req 3" in e for e in errs), errs


def test_older_dumps_are_checked_as_whole_rows(tmp_path):
    c, kq, vq = _batch()
    path, *_ = _dump(tmp_path, c, kq, vq)
    d = {k: v for k, v in debug_dump.load(path).items() if k != "source"}
    assert "tile_piece" not in d and debug_dump.check(d) == []


@pytest.mark.parametrize("interleaved", [True, False])
def test_replayed_caches_keep_shape_strides_and_storage(interleaved):
    kv = torch.zeros(6, 2, 16, 2 * 64, dtype=torch.int8)
    by_slot = kv.permute(0, 2, 1, 3)
    k, v = (by_slot[..., 64:], by_slot[..., :64]) if interleaved else (torch.zeros(6, 16, 2, 64, dtype=torch.int8),) * 2
    d = {"cache_shape": tuple(k.shape), "k_stride": k.stride(), "v_stride": v.stride(), "v_offset": -64 if interleaved else None}
    a, b = debug_dump._random_caches(d, torch.Generator().manual_seed(0), "cpu")
    assert a.shape == b.shape == k.shape and a.stride() == k.stride() and b.stride() == v.stride()
    assert (a.untyped_storage().data_ptr() == b.untyped_storage().data_ptr()) == interleaved
    assert int(a.min()) == int(b.min()) == -127 and int(a.max()) == int(b.max()) == 127
    if interleaved:
        assert b.data_ptr() + 64 == a.data_ptr()


@pytest.mark.gpu
def test_dump_of_a_real_call_replays_on_the_gpu(tmp_path, monkeypatch):
    """KVQ_DEBUG_DUMP set around a mixed-batch paged_attention call: the dump is written, its bounds report
    is clean, and the replay on the HIP prefill kernel (random tensors, the dumped metadata) matches the
    oracle on those tensors for every covered row (the reference's long-row bar, rel_l2 < 1e-2, and
    max-abs 2e-2); the replay leaves the other rows untouched."""
    c, kq, vq = _batch()
    path = str(tmp_path / "real_call.pt")
    monkeypatch.setenv("KVQ_DEBUG_DUMP", path)
    plan = ck.plan_long(c["cu"], c["seq_lens"], 16)
    dc = {k: (v.cuda() if isinstance(v, torch.Tensor) else v) for k, v in c.items()}
    st = {k: v.cuda() for k, v in c["static"].items()}
    ck.paged_attention(dc["q"], kq.cuda(), vq.cuda(), torch.empty_like(dc["q"]), dc["cu"], dc["seq_lens"],
                       dc["block_table"], 200, c["scale"], st, plan)
    torch.cuda.synchronize()
    assert os.path.exists(path)
    d = debug_dump.load(path)
    assert debug_dump.check(d) == []
    q, kt, vt, out = debug_dump.replay(d, seed=3)
    torch.cuda.synchronize()
    ref = oracle_replay(d, q, kt, vt)
    cov = ~torch.isnan(ref[:, 0, 0])
    e = O.compare(ref[cov], out.cpu()[cov])
    record("debug_dump_gpu_replay", **e)
    assert e["rel_l2"] < 1e-2 and e["max_abs"] <= 2e-2, e
    assert torch.isnan(out.cpu()[~cov].float()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("cut", [True, False])
@pytest.mark.parametrize("source", ["0", "1", "fold"])
@pytest.mark.parametrize("interleaved", [True, False])
def test_every_form_replays_as_it_ran(tmp_path, monkeypatch, cut, source, interleaved):
    """The dumps of real calls in every form the long path takes: the list on the device is the dump's, its report
    is clean, and the replay -- pieces merged, INT8 pages read where the call read them -- matches the oracle."""
    c, kq, vq = _batch()
    path = str(tmp_path / "call.pt")
    monkeypatch.setenv("KVQ_DEBUG_DUMP", path)
    monkeypatch.setenv("KVQ_PREFILL_DIRECT", source)
    _cut(monkeypatch, cut)
    if interleaved:
        kq, vq = torch.cat([kq.cuda(), vq.cuda()], -1).split(128, -1)
    plan = ck.plan_long(c["cu"], c["seq_lens"], 16)
    dc = {k: (v.cuda() if isinstance(v, torch.Tensor) else v) for k, v in c.items()}
    ck.long_attention(dc["q"], kq.cuda(), vq.cuda(), torch.empty_like(dc["q"]), dc["cu"], dc["seq_lens"], dc["block_table"],
                      200, plan, c["scale"], {k: v.cuda() for k, v in c["static"].items()})
    d = debug_dump.load(path)
    assert debug_dump.check(d) == [] and ("tile_piece" in d) == cut and d["source"] == source
    ran = {}
    for name in ("int8_prefill_attention", "paged_prefill_attention"):
        def run(*a, real=getattr(ck.ext(), name), name=name):
            ran[name] = a
            return real(*a)
        monkeypatch.setattr(ck.ext(), name, run)
    q, kt, vt, out = debug_dump.replay(d, seed=3)
    torch.cuda.synchronize()
    assert list(ran) == ["paged_prefill_attention" if source == "0" else "int8_prefill_attention"]
    if source != "0":
        _, k, v, *rest = ran["int8_prefill_attention"]
        assert k.stride() == d["k_stride"] == tuple(kq.stride()) and v.stride() == d["v_stride"] == tuple(vq.stride())
        assert rest[-2] == (source == "fold")
    ref = oracle_replay(d, q, kt, vt)
    cov = ~torch.isnan(ref[:, 0, 0])
    e = O.compare(ref[cov], out.cpu()[cov])
    record("debug_dump_forms", cut=cut, source=source, **e)
    assert e["rel_l2"] < 1e-2 and e["max_abs"] <= 2e-2, e
    assert torch.isnan(out.cpu()[~cov].float()).all()
