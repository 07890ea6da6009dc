"""Batches that leave the chip idle: fewer pieces of work than workgroups (attn_kernel, verify_kernel)."""
import pytest
import torch
from conftest import nan_like, nan_segm

from kvq import cuda_kernels as ck
from kvq import synth
from test_gpu_kernels import _check_dequant, _random_pages, check_attention, dev, int8_cache, oracle_attention

pytestmark = pytest.mark.gpu

# key counts of the requests: from one piece of one request up to several pieces per XCD, with counts around
# multiples of the 8 XCDs (2 kv heads, worker shares of at least 4 tiles of 32 keys, fixed cost included; 8 for q_len 8)
BATCHES = {"one_tile": [1], "one_piece": [200], "three": [200, 40, 1], "eight": [256, 256, 256, 250],
           "nine": [300, 600, 33, 513], "long": [5000], "long_and_short": [7, 9000, 16, 1025]}


@pytest.mark.parametrize("batch", list(BATCHES))
@pytest.mark.parametrize("q_len", [1, 3, 8])
def test_workgroup_order_of_small_batches(batch, q_len, monkeypatch):
    """The XCD-aware order hands the workers that hold units to the workgroups of all 8 XCDs; every worker must
    run exactly once, so the output equals the plain order's (worker = block) bit for bit."""
    lens = [max(n, q_len) for n in BATCHES[batch]]
    params = synth.channel_params(2, 128)
    c = synth.paged_case(14, 2, [q_len] * len(lens), lens, seed=40 + q_len, params=params)
    c["static"] = synth.calibration_scales(2, 128, params)
    c["scale"] = 128 ** -0.5
    kq, vq = int8_cache(c)
    d = dev(c)
    outs = []
    for order in ("1", "0"):
        monkeypatch.setenv("KVQ_XCD_ORDER", order)
        outs.append(ck.decode_attention(d["q"], dev(kq), dev(vq), nan_like(d["q"]), d["cu"], d["seq_lens"],
                                        d["block_table"], c["scale"], d["static"],
                                        segm=nan_segm(d["q"].shape[0], 14, 16, 128), max_query_len=q_len))
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
    check_attention(oracle_attention(c, kq, vq), outs[0], "small_batch_order", batch=batch, q_len=q_len)


@pytest.mark.parametrize("n", [1, 9, 32, 33])
@pytest.mark.parametrize("heads", [(14, 2), (2, 2), (10, 2)])
@pytest.mark.parametrize("segm", [False, True])
def test_key_splits_at_their_edges(n, heads, segm):
    """Pieces of 1 to 9 tiles around the shortest that is cut and the shortest that the key splits share (4 tiles),
    with 4 key splits (up to 64 pairs: 32 requests of 2 kv heads) and 2 (33), cut or in one pass."""
    hq, hkv = heads
    lens = [(1, 32, 33, 96, 127, 128, 129, 160, 257, 288)[i % 10] for i in range(n)]
    params = synth.channel_params(hkv, 128)
    c = synth.paged_case(hq, hkv, [1] * n, lens, seed=50 + n, params=params)
    c["static"] = synth.calibration_scales(hkv, 128, params)
    c["scale"] = 128 ** -0.5
    kq, vq = int8_cache(c)
    d = dev(c)
    out = ck.decode_attention(d["q"], dev(kq), dev(vq), nan_like(d["q"]), d["cu"], d["seq_lens"], d["block_table"],
                              c["scale"], d["static"], segm=nan_segm(n, hq, 16, 128) if segm else None)
    check_attention(oracle_attention(c, kq, vq), out, "key_split_edges", n=n, heads=list(heads), segm=segm)


@pytest.mark.parametrize("heads,q_lens", [((1, 1), [1, 8]), ((71, 1), [1, 2]), ((3, 1), [8, 5]), ((127, 1), [8])])
def test_row_to_token_division(heads, q_lens):
    """(token, q head) rows of 1, 3, 71 and 127 q heads per kv head: the row's token comes from a multiplication."""
    hq, hkv = heads
    params = synth.channel_params(hkv, 128)
    c = synth.paged_case(hq, hkv, q_lens, [300 + 7 * i for i in range(len(q_lens))], seed=60 + hq, params=params)
    c["static"] = synth.calibration_scales(hkv, 128, params)
    c["scale"] = 128 ** -0.5
    kq, vq = int8_cache(c)
    d = dev(c)
    out = ck.decode_attention(d["q"], dev(kq), dev(vq), nan_like(d["q"]), d["cu"], d["seq_lens"], d["block_table"],
                              c["scale"], d["static"], segm=nan_segm(sum(q_lens), hq, 16, 128), max_query_len=max(q_lens))
    check_attention(oracle_attention(c, kq, vq), out, "row_division", heads=list(heads))


@pytest.mark.parametrize("D,bs,pages,H", [(128, 64, 1, 8), (64, 128, 3, 5), (128, 256, 2, 3), (64, 32, 700, 16),
                                          (128, 8, 1, 2), (128, 64, 300, 8)])
@pytest.mark.parametrize("per_channel", [True, False])
def test_dequant_token_slices_bit_exact(D, bs, pages, H, per_channel):
    """Few pages: a page's tokens over several workgroups (slices of 4 tokens and up, a last one shorter)."""
    kq, vq, bt, src_req, src_j, st = _random_pages(max(pages, 4), bs, H, D, pages, pages + bs, per_channel)
    _check_dequant(kq, vq, bt, src_req, src_j, st)


@pytest.mark.parametrize("requests", [16, 17])
@pytest.mark.parametrize("q_len", [2, 3, 4, 5])
def test_row_and_pair_counts_around_the_kernel_rule(q_len, requests):
    """16, 24, 32 and 40 rows per kv head of 16 and 17 (request, kv head) pairs, cut and whole: one row tile, two
    of attn_kernel or verify_kernel, as verify_rows has it, against the oracle."""
    lens = [max(q_len, (97 * i * i + 60) % 1400) for i in range(requests)]
    params = synth.channel_params(1, 128)
    c = synth.paged_case(8, 1, [q_len] * requests, lens, seed=60 + q_len, params=params)
    c["static"] = synth.calibration_scales(1, 128, params)
    c["scale"] = 128 ** -0.5
    kq, vq = int8_cache(c)
    d, ref = dev(c), oracle_attention(c, kq, vq)
    for segm in (nan_segm(d["q"].shape[0], 8, 16, 128), None):
        out = ck.decode_attention(d["q"], dev(kq), dev(vq), nan_like(d["q"]), d["cu"], d["seq_lens"], d["block_table"],
                                  c["scale"], d["static"], segm=segm, max_query_len=q_len)
        check_attention(ref, out, "kernel_rule", requests=requests, q_len=q_len, segm=segm is not None)
