"""kvq._torch_calls against the Python path it stands for: the same results where both serve a call, and the same
error where the Python path refuses one."""
import ctypes
import threading

import pytest
import torch
from conftest import nan_like, nan_segm

from kvq import _native, synth
from kvq import cuda_kernels as ck
from test_gpu_kernels import dev, int8_cache

pytestmark = pytest.mark.gpu
HQ, HKV, D = 14, 2, 128


def _case():
    params = synth.channel_params(HKV, D)
    c = synth.paged_case(HQ, HKV, [1, 8, 40, 1, 200], [300, 1000, 40, 17, 2000], seed=77, params=params)
    c["static"] = synth.calibration_scales(HKV, D, params)
    kq, vq = int8_cache(c)
    d = dev(c)
    d.update(kc=dev(kq), vc=dev(vq), plan=ck.plan_long(c["cu"], c["seq_lens"], 16),
             slots=torch.arange(5, 5 + d["q"].shape[0], device="cuda"), key=torch.randn_like(d["q"])[:, :HKV],
             value=torch.randn_like(d["q"])[:, HKV:2 * HKV])
    return d


def _attend(d):
    out = nan_like(d["q"])
    return ck.paged_attention(d["q"], d["kc"], d["vc"], out, d["cu"], d["seq_lens"], d["block_table"], 200, D ** -0.5,
                              d["static"], d["plan"], d.get("segm"), q_group=d.get("q_group"))


def _write(d):
    kc, vc = torch.zeros_like(d["kc"]), torch.zeros_like(d["vc"])
    ck.quant_reshape_and_cache(d["key"], d["value"], kc, vc, d["slots"], d["static"])
    return torch.stack([kc, vc])


def _outcome(f, d):
    try:
        return f(d)
    except Exception as e:  # noqa: BLE001 - compared with the other path's
        return type(e), str(e)


def _both(f, d, monkeypatch):
    """The result, or (error type, text), of f with the native calls and without; and whether the native calls
    served it alone."""
    assert ck.ext().calls is not None, "kvq._torch_calls is not built"

    def python_path(*a):
        raise AssertionError("the Python path")

    with monkeypatch.context() as m:
        for op in ("quant_cache", "int8_decode_attention", "dequant_pages", "int8_prefill_attention"):
            m.setattr(ck.ext(), op, python_path)
        served = not isinstance(_outcome(f, d), tuple)
    native = _outcome(f, d)
    with monkeypatch.context() as m:
        m.setattr(ck.ext(), "calls", None)
        python = _outcome(f, d)
    return native, python, served


FORMS = {
    "plain": lambda d: {},
    "split": lambda d: {"segm": nan_segm(d["q"].shape[0], HQ, 16, D)},
    "short_split_rows": lambda d: {"segm": nan_segm(3, HQ, 4, D)},
    "strided_split": lambda d: {"segm": tuple(x[:, :HQ] for x in nan_segm(d["q"].shape[0], HQ + 2, 8, D))},
    "q_group32": lambda d: {"q_group": 32},
    "packed_q": lambda d: {"q": torch.cat([d["q"], d["q"]], 1)[:, :HQ]},
    "wide_table": lambda d: {"block_table": torch.cat([d["block_table"], d["block_table"]], 1)[:, :d["block_table"].shape[1]]},
    "scale_parameter": lambda d: {"static": {k: torch.nn.Parameter(v, requires_grad=False) for k, v in d["static"].items()}},
    "interleaved": lambda d: dict(zip(("kc", "vc"), torch.cat([d["kc"], d["vc"]], -1).transpose(1, 2).contiguous()
                                      .transpose(1, 2).split(D, -1))),
    # refused
    "q_fp16": lambda d: {"q": d["q"].half()},
    "cache_uint8": lambda d: {"kc": d["kc"].view(torch.uint8)},
    "lens_int64": lambda d: {"seq_lens": d["seq_lens"].long()},
    "host_lens": lambda d: {"seq_lens": d["seq_lens"].cpu()},
    "host_table": lambda d: {"block_table": d["block_table"].cpu()},
    "table_columns": lambda d: {"block_table": d["block_table"].repeat(1, 2)[:, ::2]},
    "scale_rows": lambda d: {"static": {**d["static"], "k_scale": d["static"]["k_scale"][:1]}},
    "scale_fp64": lambda d: {"static": {**d["static"], "v_scale": d["static"]["v_scale"].double()}},
    "odd_split": lambda d: {"segm": tuple(x.transpose(0, 1) for x in nan_segm(HQ, d["q"].shape[0], 4, D))},
    "many_splits": lambda d: {"segm": nan_segm(d["q"].shape[0], HQ, 65, D)},
    "q_group_16": lambda d: {"q_group": 16},
    "misaligned": lambda d: {"q": torch.cat([d["q"], d["q"]], 2).flatten()[4:4 + d["q"].numel()].view_as(d["q"])},
}


@pytest.mark.parametrize("direct", ["0", "1", "fold"])
@pytest.mark.parametrize("form", list(FORMS))
def test_attention_agrees_with_the_python_path(form, direct, monkeypatch):
    d = _case()
    d.update(FORMS[form](d))

    def attend(x):
        monkeypatch.setenv("KVQ_PREFILL_DIRECT", direct)
        return _attend(x)

    native, python, served = _both(attend, d, monkeypatch)
    if isinstance(python, tuple):
        assert native == python and not served
    else:
        assert served
        assert torch.equal(native.view(torch.int16), python.view(torch.int16)) and torch.isfinite(python.float()).all()


WRITES = {
    "plain": lambda d: {},
    "fewer_slots": lambda d: {"slots": d["slots"][:7]},
    "interleaved": FORMS["interleaved"],
    "no_slots": lambda d: {"slots": d["slots"][:0]},
    "slots_int32": lambda d: {"slots": d["slots"].int()},
    "slots_strided": lambda d: {"slots": d["slots"].repeat(2)[::2]},
    "more_slots": lambda d: {"slots": d["slots"].repeat(2)},
    "key_fp32": lambda d: {"key": d["key"].float()},
    "mu_rows": lambda d: {"static": {**d["static"], "k_mu": d["static"]["k_mu"][:1]}},
    "cache_heads": lambda d: {"kc": d["kc"].repeat(1, 1, 2, 1)},
    "host_slots": lambda d: {"slots": d["slots"].cpu()},
}


@pytest.mark.parametrize("form", list(WRITES))
def test_cache_write_agrees_with_the_python_path(form, monkeypatch):
    d = _case()
    d.update(WRITES[form](d))
    native, python, served = _both(_write, d, monkeypatch)
    if isinstance(python, tuple):
        assert native == python and not served
    else:
        assert served or form == "no_slots"
        assert torch.equal(native, python)


def test_streams_and_threads():
    """Calls on the current stream of their thread, from several threads at once, each with its own buffers."""
    d = _case()
    d["segm"] = None
    want = _attend(d)
    torch.cuda.synchronize()
    got, errors = {}, []

    def work(i):
        try:
            s = torch.cuda.Stream()
            with torch.cuda.stream(s):
                for _ in range(10):
                    x = dict(d, segm=nan_segm(d["q"].shape[0], HQ, 8, D))
                    got[i] = _attend(x)
            s.synchronize()
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not errors
    for i in range(3):
        assert (got[i].float() - want.float()).abs().max() < 2e-2


@pytest.mark.parametrize("failing", ["kvq_quant_cache", "kvq_int8_decode_attention", "kvq_int8_decode_attention_ex",
                                     "kvq_dequant_pages", "kvq_paged_prefill_attention", "kvq_paged_prefill_attention_ex",
                                     "kvq_int8_prefill_attention", "kvq_int8_prefill_attention_ex"])
def test_launch_errors_name_the_entry_point(failing, monkeypatch):
    """A launch the HIP runtime refuses raises what the Python path raises: entry points that return
    KVQ_ERR_LAUNCH without launching stand in for the library's, in the native module and in ctypes."""
    d = _case()
    refuse, accept = (ctypes.CFUNCTYPE(ctypes.c_int)(lambda rc=rc: rc) for rc in (_native.ERR_LAUNCH, 0))
    # (uncut work lists go to the _ex entry points too, without their lists)
    refused = {failing, failing.replace("_attention", "_attention_ex") if "prefill" in failing else failing}
    lib = _native.load()
    real = {name: ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in _native.SIGNATURES}
    stubs = {name: refuse if name in refused else accept for name in real}
    if "decode" in failing:    # fewer rows than tokens, or one each
        d["segm"] = nan_segm(3 if failing.endswith("_ex") else d["q"].shape[0], HQ, 4, D)
    if "prefill" in failing or "dequant" in failing:
        monkeypatch.setenv("KVQ_PREFILL_DIRECT", "1" if "int8" in failing else "0")
        # cut or whole: where the estimate of a merge is small or large
        cut = failing.endswith("_ex")
        monkeypatch.setattr(ck, "_prefill_us", lambda longest, groups, partials, *a: (partials is None) == cut)

    class Lib:
        kvq_last_error = staticmethod(lambda: b"no such luck")
        kvq_prefill_rows_per_tile, kvq_prefill_max_parts = lib.kvq_prefill_rows_per_tile, lib.kvq_prefill_max_parts

        def __getattr__(self, name):
            return lambda *a: _native.ERR_LAUNCH if name == failing else 0

    f = _write if failing == "kvq_quant_cache" else _attend
    ck.ext()
    try:
        ck.ext().calls.bind({name: ctypes.cast(s, ctypes.c_void_p).value for name, s in stubs.items()})
        monkeypatch.setattr(_native, "_LIB", Lib())
        native = _outcome(f, d)
        monkeypatch.setattr(ck.ext(), "calls", None)
        python = _outcome(f, d)
    finally:
        monkeypatch.undo()
        ck.ext().calls.bind(real)
    assert native == python == (_native.NativeError, f"{failing}: no such luck")
