"""Which form of the long requests' attention a call takes (long_attention, no KVQ_PREFILL_DIRECT): the INT8 pages
read by one kernel, or the two kernels -- by calls recorded in place of the kernels. No GPU."""
import numpy as np
import pytest
import torch

from kvq import cuda_kernels as ck


class Recorder:
    calls = None
    prefill_rows, prefill_max_parts = 128, 64

    def __init__(self):
        self.ran = []

    def int8_prefill_attention(self, *a):
        self.ran.append("direct")

    def dequant_pages(self, *a):
        self.ran.append("dequant")

    def paged_prefill_attention(self, *a):
        self.ran.append("prefill")


def _forms(monkeypatch, k_strides, v_strides, q_len=20, keys=40, hq=28, hkv=4, d=128, bs=16):
    e = Recorder()
    monkeypatch.setattr(ck, "_EXT", e)
    monkeypatch.delenv("KVQ_PREFILL_DIRECT", raising=False)
    nb = -(-keys // bs)
    kc, vc = (torch.empty_strided((nb, bs, hkv, d), s, dtype=torch.int8, device="meta") for s in (k_strides, v_strides))
    plan = ck.plan_long(np.array([0, q_len]), np.array([keys]), bs)
    q = torch.zeros(q_len, hq, d, dtype=torch.bfloat16)
    cu, sl = torch.tensor([0, q_len], dtype=torch.int32), torch.tensor([keys], dtype=torch.int32)
    bt = torch.zeros(1, nb, dtype=torch.int32)
    st = {"k_scale": torch.ones(hkv, 1), "v_scale": torch.ones(hkv, 1)}
    ck.long_attention(q, kc, vc, torch.empty_like(q), cu, sl, bt, q_len, plan, d ** -0.5, st)
    return e.ran


PAGE = (16 * 512, 512, 128, 1)


def test_few_rows_read_the_int8_pages(monkeypatch):
    assert _forms(monkeypatch, PAGE, PAGE) == ["direct"]


@pytest.mark.parametrize("wide", [(1 << 32, 512, 128, 1), (1 << 31, 1 << 27, 128, 1)])
@pytest.mark.parametrize("which", ["k", "v"])
def test_pages_past_the_direct_kernels_offsets_take_the_two_kernels(wide, which, monkeypatch):
    """Page strides from 4 GiB on, or slots 2 GiB apart over a page: dequant_pages takes them, the direct kernel's
    32-bit page and slot offsets do not."""
    ran = _forms(monkeypatch, wide if which == "k" else PAGE, wide if which == "v" else PAGE)
    assert ran == ["dequant", "prefill"]


def test_the_last_page_stride_the_direct_kernel_takes(monkeypatch):
    last = (1 << 32) - 16
    assert _forms(monkeypatch, (last, 512, 128, 1), (last, (1 << 27) - 16, 128, 1)) == ["direct"]


def test_lists_made_before_a_capture_serve_it(monkeypatch):
    """A program that copied a plan's lists to the device itself (gpu, tiles) before it captures the call: nothing
    may be copied inside the capture, so those lists serve it (whole rows, the two kernels)."""
    e = Recorder()
    monkeypatch.setattr(ck, "_EXT", e)
    plan = ck.plan_long(np.array([0, 20]), np.array([5000]), 16)
    plan.gpu("cpu")
    tiles = plan.tiles(7, "cpu")
    monkeypatch.setattr(ck, "_capturing", lambda device: True)
    monkeypatch.setattr(ck, "_to_device", lambda *a: pytest.fail("a copy inside the capture"))
    work = plan.work(7, 4, 128, torch.device("cpu"))
    assert work.tile_req is tiles[0] and work.tile_row is tiles[1] and work.tile_piece is None and not work.direct
    monkeypatch.undo()
    monkeypatch.setattr(ck, "_EXT", e)
    assert plan.work(7, 4, 128, torch.device("cpu")).tile_piece is not None     # outside it: the call's own list


# (q heads, kv heads, head_dim, block, "query:keys ..."): us in a graph of whole rows from the temporary cache and from
# the INT8 pages, and of cut rows from each
MEASURED = {
    (14, 2, 64, 16, "25:25 374:396 774:774"): (20.7, 23.2, 25.4, 23.8),
    (14, 2, 64, 16, "74:74 1146:1146 708:711"): (26.7, 31.6, 30.0, 29.1),
    (12, 2, 128, 16, "174:174 885:885"): (28.2, 34.6, 30.9, 30.4),
    (12, 2, 128, 16, "817:831"): (26.9, 32.3, 31.4, 30.7),
    (14, 2, 64, 32, "574:681 1196:1228"): (28.3, 33.3, 31.8, 30.3),
    (12, 2, 128, 64, "108:291"): (16.5, 17.5, 17.1, 16.4),
    (14, 2, 64, 32, "464:467"): (15.8, 16.6, 16.1, 14.2),
    (32, 8, 128, 64, "10:346"): (15.9, 16.5, 15.7, 14.0),
    (32, 8, 128, 16, "1347:1347"): (50.1, 58.9, 47.0, 51.7),
    (12, 2, 128, 16, "3931:3931"): (98.4, 135.9, 86.8, 115.0),
    (16, 16, 64, 64, "679:15047"): (244.5, 334.7, 100.9, 109.6),
    (14, 2, 64, 64, "11:4851 90:90 359:359"): (79.7, 110.8, 20.3, 17.6),
    (32, 8, 128, 16, "23:6531"): (143.5, 207.0, 36.9, 28.4),
    (28, 4, 128, 16, "118:5494"): (118.2, 176.0, 38.2, 36.8),
    (28, 4, 128, 16, "1216:1216"): (39.2, 47.4, 40.5, 43.1),
    (28, 4, 128, 16, "356:359"): (17.9, 18.5, 22.3, 21.0),
}


@pytest.mark.parametrize("step", list(MEASURED))
def test_the_form_taken_is_about_the_fastest(step):
    """The rule (split_rows, direct_pays) on measured steps: at most 10% over the fastest form, and never more than
    3% over whole rows in two kernels, which every step can run."""
    hq, hkv, d, block, chunks = step
    q, keys = zip(*(map(int, c.split(":")) for c in chunks.split()))
    plan = ck.plan_long(np.concatenate([[0], np.cumsum(q)]), np.array(keys), block)
    work = plan.work(hq // hkv, hkv, d, torch.device("cpu"))
    us = MEASURED[step]
    taken = us[2 * (work.tile_piece is not None) + work.direct]
    assert taken <= 1.1 * min(us) and taken <= 1.03 * us[0]


def test_other_head_sizes_are_refused_as_before():
    plan = ck.plan_long(np.array([0, 20]), np.array([500]), 16)
    q = torch.zeros(20, 8, 96, dtype=torch.bfloat16)
    kc = torch.zeros(32, 16, 2, 96, dtype=torch.int8)
    with pytest.raises(RuntimeError):
        ck.long_attention(q, kc, kc, torch.zeros_like(q), None, None, None, 20, plan, 1.0, {"k_scale": None, "v_scale": None})
