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
