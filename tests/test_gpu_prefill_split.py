"""The prefill kernels with a split work list (kvq_paged_prefill_attention_ex, kvq_int8_prefill_attention_ex):
rows' keys cut into pieces and merged. Checked against fp32 attention over the same pages at the bar of
test_gpu_prefill.py; the bf16 and INT8 sources cut alike must agree bit for bit."""
import numpy as np
import pytest
import torch
from conftest import nan_like, record

from oracle import kvq_oracle as O
from kvq import cuda_kernels as ck
from test_gpu_kernels import dev
from test_gpu_prefill import _reference, _temp_cache

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _split(plan, group, hkv, d, parts):
    """A work list that cuts every row tile into exactly `parts` pieces (also more than it has tiles)."""
    rows = ck.ext().prefill_rows
    req, row, _ = plan._row_tiles(group, rows)
    n = req.shape[0]
    at = np.repeat(np.arange(n), parts)
    part = np.arange(n * parts) % parts
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x, dtype=np.int32)).to(DEV)  # noqa: E731
    merge = np.stack([req, row, np.arange(n) * parts, np.full(n, parts)], 1) if parts > 1 else np.zeros((0, 4))
    nan = float("nan")
    return t(req[at]), t(row[at]), (t(part | parts << 16), t(np.arange(n * parts)), t(merge),
                                    torch.full((n * parts, hkv, rows, d), nan, device=DEV),
                                    torch.full((n * parts, hkv, rows, 2), nan, device=DEV))


@pytest.mark.parametrize("shape", [(28, 4, 128), (14, 2, 64)])
@pytest.mark.parametrize("parts", [1, 2, 3, 7, 64])
@pytest.mark.parametrize("jump", [False, True])
def test_split_prefill_matches_fp32_reference(shape, parts, jump):
    """Pieces of one tile, of none (64 pieces of rows with 4 tiles) and of several; with `jump`, keys far past
    their piece's first tile whose scores send that piece alone to the rescaling pass."""
    hq, hkv, d = shape
    q_lens, seq_lens = [100, 3, 37, 9, 200], [100, 50, 517, 2000, 1000]
    cu, plan, kt, vt = _temp_cache(q_lens, seq_lens, hkv, d, 16, seed=hq + parts)
    T = int(cu[-1])
    q = (torch.randn(T, hq, d, generator=torch.Generator().manual_seed(1)) * 2).to(torch.bfloat16)
    if jump:
        q = (q.float() * 0.5 + 0.5).to(torch.bfloat16)
        first = {r: p for p, r in reversed(list(enumerate(plan.src_req.tolist())))}
        for r, key in ((2, 250), (3, 1990), (4, 850)):
            kt[first[r] + key // 16, key % 16] = 60.0
    scale = d ** -0.5
    out = nan_like(q.to(DEV))
    _, _, bt = plan.gpu(DEV)
    tile_req, tile_row, split = _split(plan, hq // hkv, hkv, d, parts)
    ck.ext().paged_prefill_attention(q.to(DEV), kt.to(DEV), vt.to(DEV), out, cu.to(DEV),
                                     torch.tensor(seq_lens, dtype=torch.int32, device=DEV), bt, tile_req, tile_row, scale,
                                     split)
    out = out.cpu()
    ref = _reference(q, kt, vt, cu, seq_lens, plan, scale)
    got = torch.stack([out[int(cu[r]) + t] for (r, t) in ref]).float()
    err = O.compare(torch.stack(list(ref.values())), got)
    record("prefill_split", shape=list(shape), parts=parts, jump=jump, **err)
    assert torch.isfinite(got).all() and err["max_abs"] <= 2e-2 and err["mean_abs"] <= 2e-3 and err["rel_l2"] < 1e-2, err
    assert torch.isnan(out[int(cu[1]):int(cu[2])].float()).all()          # the short request's rows


@pytest.mark.parametrize("d,layout", [(128, "pages"), (128, "consecutive"), (64, "pages")])
@pytest.mark.parametrize("upper", [0, 300])
def test_split_direct_prefill_bit_identical(d, layout, upper, monkeypatch):
    """long_attention with its own split: few rows over many keys, pages in random order or consecutive (read
    without the block table, from a piece's first page on), host lengths that overstate the keys (trailing
    pieces find fewer or no tiles); both sources bit for bit, and the split against the whole rows."""
    hq, hkv, bs = (28, 4, 16) if d == 128 else (14, 2, 32)
    q_lens, seq_lens = [20, 1, 64], [3001, 40, 2100]
    g = torch.Generator().manual_seed(5)
    width = [-(-(n + upper) // bs) for n in seq_lens]
    nb = sum(width) + 4
    kq = torch.randint(-127, 128, (nb, bs, hkv, d), generator=g, dtype=torch.int8)
    vq = torch.randint(-127, 128, (nb, bs, hkv, d), generator=g, dtype=torch.int8)
    ids = torch.arange(nb) if layout == "consecutive" else torch.randperm(nb, generator=g)
    bt = torch.zeros(3, max(width), dtype=torch.int32)
    for r, n in enumerate(width):
        bt[r, :n] = ids[sum(width[:r]):sum(width[:r]) + n]
    st = {"k_scale": torch.rand(hkv, d, generator=g) * 0.02 + 1e-3, "v_scale": torch.rand(hkv, d, generator=g) * 0.02}
    cu = torch.tensor(np.concatenate([[0], np.cumsum(q_lens)]), dtype=torch.int32)
    sl = torch.tensor(seq_lens, dtype=torch.int32)
    q = torch.randn(int(cu[-1]), hq, d, generator=g).to(torch.bfloat16)
    outs = {}
    for mode, whole in (("0", 1.5), ("1", 1.5), ("0", 0)):
        monkeypatch.setenv("KVQ_PREFILL_DIRECT", mode)
        monkeypatch.setattr(ck, "PREFILL_WHOLE", whole)
        plan = ck.plan_long(cu, sl + upper, bs)
        assert (plan.work(hq // hkv, hkv, d, torch.device(DEV)).tile_piece is not None) == (whole > 0)
        out = nan_like(dev(q))
        ck.long_attention(dev(q), dev(kq), dev(vq), out, dev(cu), dev(sl), dev(bt), 64, plan, d ** -0.5, dev(st))
        outs[mode, whole] = out.cpu()
    long_rows = torch.repeat_interleave(torch.tensor(q_lens) > ck.SHORT_Q, torch.tensor(q_lens))
    assert torch.equal(outs["0", 1.5].view(torch.int16), outs["1", 1.5].view(torch.int16))
    err = O.compare(outs["0", 0][long_rows], outs["0", 1.5][long_rows])
    assert err["max_abs"] <= 2e-2 and err["rel_l2"] < 5e-3, err            # bf16 P and output, sums in another order


def _both_orders(src, hq, hkv, d, q_len, ids, parts, seed):
    """One request over the pages `ids` (in this order) of a contiguous cache, cut into `parts` pieces, and the same
    keys with the pages in another order, read through the block table: (out, out)."""
    n = ids.shape[0]
    g = torch.Generator(device=DEV).manual_seed(seed)
    shape = (n, 16, hkv, d)
    if src == "int8":
        k, v = (torch.randint(-127, 128, shape, generator=g, device=DEV, dtype=torch.int8) for _ in range(2))
    else:
        k, v = (torch.randn(shape, generator=g, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    st = [torch.rand(hkv, d, generator=g, device=DEV) * 0.02 + 1e-3 for _ in range(2)]
    q = torch.randn(q_len, hq, d, generator=g, device=DEV, dtype=torch.bfloat16)
    cu = torch.tensor([0, q_len], dtype=torch.int32, device=DEV)
    sl = torch.tensor([16 * n - 3], dtype=torch.int32, device=DEV)
    plan = ck.plan_long(np.array([0, q_len]), np.array([16 * n - 3]), 16)
    tile_req, tile_row, split = _split(plan, hq // hkv, hkv, d, parts)
    outs = []
    for swap in (False, True):
        if swap:    # a page moves to another place: pages i and n - 1 - i trade places, the table follows
            k, v, ids = k.flip(0).contiguous(), v.flip(0).contiguous(), n - 1 - ids
        out = nan_like(q)
        args = (q, k, v, out, cu, sl, ids.to(device=DEV, dtype=torch.int32)[None].contiguous(), tile_req, tile_row, d ** -0.5)
        if src == "int8":
            ck.ext().int8_prefill_attention(*args, *st, split=split if parts > 1 else None)
        else:
            ck.ext().paged_prefill_attention(*args, split=split if parts > 1 else None)
        outs.append(out)
    return outs


@pytest.mark.parametrize("src", ["bf16", "int8"])
def test_piece_of_pages_with_low_ids(src):
    """Pieces whose consecutive pages have ids below their place in the request: the run's key 0 would lie before
    the cache. The last 63 pages are pages 0 .. 62, the 62 before them lie after those in a scattered order."""
    ids = torch.cat([63 + (torch.arange(62) * 23) % 62, torch.arange(63)])
    a, b = _both_orders(src, 28, 4, 128, 40, ids, 7, 1)
    assert torch.isfinite(a.float()).all() and torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("parts", [1, 64])
@pytest.mark.parametrize("src,hkv", [("bf16", 32), ("int8", 64)])
def test_run_of_pages_longer_than_4_gib(src, hkv, parts):
    """532,480 keys on consecutive pages, 4.06 GiB of K from the first key to the last: the offset of a key within
    the run needs more than 32 bits."""
    a, b = _both_orders(src, hkv, hkv, 128, 12, torch.arange((1 << 15) + 512), parts, 2)
    assert torch.isfinite(a.float()).all() and torch.equal(a.view(torch.int16), b.view(torch.int16))


def test_capture_after_the_plans_own_copies(monkeypatch):
    """A program that made the plan's device copies itself (gpu, tiles) and then captures its first call: the graph
    holds the whole rows' two kernels; replays follow the inputs, and a later eager call agrees."""
    monkeypatch.delenv("KVQ_PREFILL_DIRECT", raising=False)
    g = torch.Generator().manual_seed(9)
    nb, hq, hkv, d = 160, 28, 4, 128
    kq, vq = (torch.randint(-127, 128, (nb, 16, hkv, d), generator=g, dtype=torch.int8).to(DEV) for _ in range(2))
    st = {k: (torch.rand(hkv, d, generator=g) * 0.02 + 1e-3).to(DEV) for k in ("k_scale", "v_scale")}
    q = torch.randn(20, hq, d, generator=g).to(torch.bfloat16).to(DEV)
    cu, sl = (torch.tensor(x, dtype=torch.int32, device=DEV) for x in ([0, 20], [2500]))
    bt = torch.randperm(nb, generator=g)[None].to(torch.int32).to(DEV)
    plan = ck.plan_long(np.array([0, 20]), np.array([2500]), 16)
    plan.gpu(DEV)
    plan.tiles(hq // hkv, DEV)
    out = nan_like(q)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ck.long_attention(q, kq, vq, out, cu, sl, bt, 20, plan, d ** -0.5, st)
    for i in range(3):
        q.normal_()
        out.fill_(float("nan"))
        graph.replay()
        want = ck.long_attention(q, kq, vq, nan_like(q), cu, sl, bt, 20, plan, d ** -0.5, st)
        err = O.compare(want.cpu(), out.cpu())
        assert torch.isfinite(out.float()).all() and err["max_abs"] <= 2e-2 and err["rel_l2"] < 5e-3, (i, err)
