"""decode_attention's native call path (_dk_native) against its Python path: the same bits where
it takes a call, and the Python path's result or error for every call that it leaves."""
import sys
import warnings
from types import SimpleNamespace

import pytest
import torch

import _dk_native
import attention
import layout
from attention import decode_attention

DEV = "cuda"


def _python_only(monkeypatch):
    monkeypatch.setattr(attention, "_NATIVE", lambda *a: None)


def _inputs(dtype=torch.float16, fp8=False, hq=8, hkv=2, d=64, lens=(40, 0, 17)):
    q, kv, indptr, ids, last, _ = layout.synthesize_paged(
        len(lens), list(lens), hq, hkv, d, dtype=dtype, device=DEV, page_table="permuted", seed=2)
    return q, kv.to(torch.float8_e4m3fn) if fp8 else kv, indptr, ids, last


FORMS = {
    "plain": lambda a: (a, {}),
    "automatic, hinted": lambda a: (a + (None,), dict(max_pages_per_seq=3)),
    "split": lambda a: (a + (4,), {}),
    "pair": lambda a: ((a[0], (a[1][:, 0], a[1][:, 1])) + a[2:], {}),
    "pair as a list": lambda a: ((a[0], [a[1][:, 0], a[1][:, 1]]) + a[2:] + (0,), {}),
    "options": lambda a: (a + (2,), dict(sm_scale=0.3, logit_cap=7.0, window=9,
                                         sinks=torch.linspace(-1, 1, a[0].shape[1], device=DEV))),
    "off by zero": lambda a: (a, dict(logit_cap=0.0, window=0)),
    "integer scale": lambda a: (a, dict(sm_scale=1)),
    "strided q and out": lambda a: (
        (torch.cat([a[0], a[0]], 1)[:, :a[0].shape[1]],) + a[1:],
        dict(out=torch.empty(a[0].shape[0], 2 * a[0].shape[1], a[0].shape[2], dtype=a[0].dtype,
                             device=DEV)[:, ::2])),
    "own workspace": lambda a: (a + (0,), dict(workspace=torch.empty(64 << 20, dtype=torch.uint8,
                                                                     device=DEV))),
    "strided tables": lambda a: (a[:2] + tuple(t.repeat_interleave(2)[::2] for t in a[2:]), {}),
    "32-token pages": lambda a: (
        (a[0], torch.cat([a[1], a[1]], 2)) + a[2:4] + (a[4],), {}),
}


@pytest.mark.gpu
@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("dtype,fp8", [(torch.float16, False), (torch.bfloat16, True)])
def test_same_bits_as_the_python_path(monkeypatch, form, dtype, fp8):
    print(f"[case] native {form} {dtype} fp8={fp8}", flush=True)
    if fp8 and form == "32-token pages":
        pytest.skip("torch has no cat of fp8 tensors on the GPU")
    args, kw = FORMS[form](_inputs(dtype, fp8))
    if fp8:
        kw = dict(kw, k_scale=0.5, v_scale=2.0)
    got = decode_attention(*args, **kw).clone()
    _python_only(monkeypatch)
    want = decode_attention(*args, **kw)
    torch.cuda.synchronize()
    assert got.dtype == want.dtype and torch.equal(got, want)


BAD = {
    "page table on the host": lambda a: (a[:2] + (a[2].cpu(),) + a[3:], {}),
    "int64 table": lambda a: (a[:3] + (a[3].long(),) + a[4:], {}),
    "float32 q": lambda a: ((a[0].float(),) + a[1:], {}),
    "heads": lambda a: ((a[0][:, :3],) + a[1:], {}),
    "head_dim stride": lambda a: ((a[0].transpose(1, 2).contiguous().transpose(1, 2),) + a[1:], {}),
    "batch": lambda a: ((a[0][:2],) + a[1:], {}),
    "negative split": lambda a: (a + (-1,), {}),
    "boolean split": lambda a: (a + (True,), {}),
    "huge split": lambda a: (a + (1 << 20,), {}),
    "scale": lambda a: (a, dict(sm_scale=float("nan"))),
    "fp8 scale on fp16": lambda a: (a, dict(k_scale=0.5)),
    "cap": lambda a: (a, dict(logit_cap=-1.0)),
    "window": lambda a: (a, dict(window=-3)),
    "sinks": lambda a: (a, dict(sinks=torch.zeros(3, device=DEV))),
    "out": lambda a: (a, dict(out=torch.empty_like(a[0][:2]))),
    "workspace": lambda a: (a + (4,), dict(workspace=torch.empty(16, dtype=torch.uint8,
                                                                 device=DEV))),
    "unaligned q": lambda a: ((torch.empty(a[0].numel() + 1, dtype=a[0].dtype,
                                           device=DEV)[1:].view_as(a[0]),) + a[1:], {}),
    "not a tensor": lambda a: (a[:4] + ([1, 2, 3],), {}),
    "option out of range": lambda a: (a, dict(qk_path=9)),
}


@pytest.mark.gpu
@pytest.mark.parametrize("what", list(BAD))
def test_same_errors_as_the_python_path(monkeypatch, what):
    args, kw = BAD[what](_inputs())
    attention._PLANS.clear()             # True == 1: a plan kept for split 1 would take it
    with pytest.raises((ValueError, RuntimeError, TypeError)) as got:
        decode_attention(*args, **kw)
    _python_only(monkeypatch)
    attention._PLANS.clear()
    with pytest.raises((ValueError, RuntimeError, TypeError)) as want:
        decode_attention(*args, **kw)
    assert type(got.value) is type(want.value) and str(got.value) == str(want.value)


@pytest.mark.gpu
def test_scratch_is_the_librarys_and_follows_the_stream():
    args = _inputs(lens=(700, 900, 33))
    base = decode_attention(*args, 4)
    keys = set(attention._SCRATCH._by_stream)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        out = decode_attention(*args, 4)
    torch.cuda.synchronize()
    assert torch.equal(out, base)
    assert set(attention._SCRATCH._by_stream) - keys == {(torch.device("cuda", 0), s.cuda_stream)}


def test_left_to_python_without_a_gpu():
    attention._bind_native()
    q, kv, indptr, ids, last, _ = layout.synthesize(2, 16, 4, 2, 64, device="cpu")
    call = (q, kv, indptr, ids, last, 1, None, None, 0, 0, 0, 0, 0) + (None,) * 6
    assert _dk_native.decode(*call) is None
    assert _dk_native.decode(*(None,) * 19) is None
    with pytest.raises(TypeError):
        _dk_native.decode(q)


def _refuse_bind(*args):
    raise AssertionError("bound an extension that does not fit")


def _other(at, value):
    built = list(_dk_native.BUILT_FOR)
    built[at] = value
    return SimpleNamespace(BUILT_FOR=tuple(built), bind=_refuse_bind, decode=_refuse_bind)


# missing, too old to say what it fits, another interface version, struct size, torch, Python
UNUSABLE = [None, SimpleNamespace(bind=_refuse_bind), _other(0, 2), _other(1, 48), _other(2, 56),
            _other(3, "2.9.1"), _other(5, 9)]


@pytest.mark.parametrize("module", UNUSABLE)
def test_an_extension_that_does_not_fit_leaves_every_call_to_python(monkeypatch, module):
    monkeypatch.setattr(attention, "_NATIVE", None)
    monkeypatch.setitem(sys.modules, "_dk_native", module)
    with pytest.warns(RuntimeWarning, match="__graft_entry__.py build"):
        bound = attention._bind_native()
    assert attention._NATIVE is bound and bound(*range(19)) is None


def test_the_built_extension_fits(monkeypatch):
    monkeypatch.setattr(attention, "_NATIVE", None)
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert attention._bind_native() is _dk_native.decode


@pytest.mark.gpu
def test_calls_run_without_the_extension(monkeypatch):
    args = _inputs()
    want = decode_attention(*args, 4)
    monkeypatch.setattr(attention, "_NATIVE", None)
    monkeypatch.setitem(sys.modules, "_dk_native", None)
    with pytest.warns(RuntimeWarning):
        got = decode_attention(*args, 4)
    with warnings.catch_warnings():       # said once
        warnings.simplefilter("error")
        assert torch.equal(decode_attention(*args, 4), want) and torch.equal(got, want)
