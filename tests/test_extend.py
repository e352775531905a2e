"""Extend (prefill) attention on the HIP kernel against the backend's PyTorch path.

The kernel and the PyTorch path take the same bf16 / fp16 inputs, compute in fp32 and round
once, so their outputs may differ by one unit in the last place of the output type (2^-10 of
the value in fp16, 2^-7 in bf16) plus what fp32 sums over the longest context differ by (1e-5).
"""
import ctypes
import math

import pytest
import torch

import dk_lib
import extend
import sglang_backend
from sglang_fakes import make_batch

DEV = "cuda"
ULP = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}


def _batch(new, pre, hq, hkv, d, dtype, cache=None, seed=0, cap=None, win=None, device=DEV):
    lens = [n + p for n, p in zip(new, pre)]
    sc = dict(k_scale=0.5, v_scale=0.25) if cache is not None else {}
    fb, layers, pool, r2t = make_batch(lens, hq=hq, hkv=hkv, d=d, layers=1, dtype=dtype,
                                       device=device, seed=seed, decode=False, kv_dtype=cache,
                                       **sc)
    layer = layers[0]
    layer.logit_cap = cap
    layer.sliding_window_size = -1 if win is None else win - 1
    rows = fb.req_pool_indices.tolist()
    fb.out_cache_loc = torch.cat([r2t[r, n - m:n] for r, n, m in zip(rows, lens, new)]).long().to(
        device)
    fb.extend_seq_lens_cpu = list(new)
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    t = sum(new)
    qkv = torch.randn(t, hq + 2 * hkv, d, generator=g, device=device).to(dtype)
    return fb, layer, pool, qkv


def _both(monkeypatch, fb, layer, q, k, v, **kw):
    """(kernel path, PyTorch path), the first checked to have been the kernel's."""
    backend = sglang_backend.SplitKVHipBackend()
    used = []
    real = extend.extend_attention
    with monkeypatch.context() as m:
        m.setattr(extend, "extend_attention", lambda *a, **b: used.append(1) or real(*a, **b))
        got = backend.forward_extend(q, k, v, layer, fb, **kw)
        torch.cuda.synchronize()
    assert used == [1]
    with monkeypatch.context() as m:
        m.setattr(extend, "takes", lambda *a: False)
        want = backend.forward_extend(q, k, v, layer, fb, **kw)
    return got, want


def _close(got, want):
    assert got.shape == want.shape and got.dtype == want.dtype
    d = (got.float() - want.float()).abs()
    assert bool((d <= ULP[got.dtype] * want.float().abs() + 1e-5).all()), float(d.max())


# query rows around a wavefront's 32 and a workgroup's 128, keys around the tiles' 32 and 64,
# a single token, one without a prefix, one empty request
SIZES = [([1], [0]), ([1, 33, 0, 8], [63, 0, 5, 64]), ([32, 31, 129], [0, 33, 1]),
         ([200], [311]), ([7, 65], [121, 127])]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("heads", [(8, 8), (32, 8), (28, 4), (16, 1)])
def test_sizes_and_groups(monkeypatch, dtype, d, heads):
    hq, hkv = heads
    for i, (new, pre) in enumerate(SIZES):
        print(f"[case] extend {dtype} d={d} {hq}/{hkv} new={new} pre={pre}", flush=True)
        fb, layer, pool, qkv = _batch(new, pre, hq, hkv, d, dtype, seed=i)
        q, k, v = qkv.split([hq, hkv, hkv], dim=1)          # strided views of a fused projection
        got, want = _both(monkeypatch, fb, layer, q.reshape(-1, hq * d) if i % 2 else q, k, v)
        _close(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("cache", [None, torch.float8_e4m3fn])
@pytest.mark.parametrize("cap,win,sinks", [(None, 1, False), (None, 70, False), (20.0, None, False),
                                           (None, None, True), (5.0, 33, True)])
@pytest.mark.parametrize("dtype,d", [(torch.float16, 64), (torch.bfloat16, 128),
                                     (torch.float16, 256)])
def test_options(monkeypatch, cache, cap, win, sinks, dtype, d):
    print(f"[case] extend options {dtype} d={d} cache={cache} cap={cap} win={win} sinks={sinks}",
          flush=True)
    fb, layer, pool, qkv = _batch([150, 3, 40], [10, 200, 0], 16, 4, d, dtype, cache, cap=cap,
                                  win=win, seed=3)
    q, k, v = (t.contiguous() for t in qkv.split([16, 4, 4], dim=1))
    kw = {"sinks": torch.randn(16, device=DEV)} if sinks else {}
    got, want = _both(monkeypatch, fb, layer, q, k, v, **kw)
    _close(got, want)


@pytest.mark.gpu
def test_many_requests_and_long_context(monkeypatch):
    # more requests than one launch takes; then one long prefix (many key tiles per workgroup)
    n = 300
    fb, layer, pool, qkv = _batch([1 + i % 3 for i in range(n)], [i % 40 for i in range(n)], 4, 2,
                                  64, torch.bfloat16, seed=5)
    q, k, v = (t.contiguous() for t in qkv.split([4, 2, 2], dim=1))
    _close(*_both(monkeypatch, fb, layer, q, k, v))
    fb, layer, pool, qkv = _batch([70], [4000], 8, 2, 128, torch.float16, seed=6)
    q, k, v = (t.contiguous() for t in qkv.split([8, 2, 2], dim=1))
    _close(*_both(monkeypatch, fb, layer, q, k, v))


def _direct(q, kp, vp, r2t, rows, new, pre, workspace=True, win=None, sinks=None):
    """The C ABI's call with its workspace, without one (False), or with one that it cannot use
    ("short", "unaligned"); returns (out, the workspace's bytes)."""
    t, hq, d = q.shape
    hkv, n = kp.shape[1], len(new)
    ints = ctypes.c_int32 * n
    lib = dk_lib.load()
    news, alls = ints(*new), ints(*(a + b for a, b in zip(new, pre)))
    out = torch.full_like(q, float("nan"))
    need = lib.dk_extend_workspace_bytes(n, news, alls, hq, hkv, d, win or 0)
    ws = torch.empty(need + 256, dtype=torch.uint8, device=q.device)
    at, size = {True: (ws.data_ptr(), need), False: (None, 0), "short": (ws.data_ptr(), need - 1),
                "unaligned": (ws.data_ptr() + 16, need)}[workspace]
    s = dk_lib.DkExtendStrides(q.stride(0), d, kp.stride(0), d, vp.stride(0), d, out.stride(0), d)
    rc = lib.dk_extend_attention(
        q.data_ptr(), kp.data_ptr(), vp.data_ptr(), r2t.data_ptr(), r2t.stride(0), r2t.shape[0],
        ints(*rows), news, alls, out.data_ptr(), at, size, n, t, hq, hkv, d, kp.shape[0],
        0 if q.dtype == torch.float16 else 1, dk_lib.DK_KV_SAME, ctypes.byref(s), d ** -0.5, 1.0,
        0.0, win or 0, None if sinks is None else sinks.data_ptr(),
        torch.cuda.current_stream().cuda_stream)
    dk_lib.check(rc, "dk_extend_attention")
    return out, need


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,d", [(torch.float16, 64), (torch.bfloat16, 128),
                                     (torch.bfloat16, 256)])
@pytest.mark.parametrize("new,pre,win,sinks", [
    ([1], [4000], None, False), ([16, 3], [3000, 10], None, True), ([40], [600], None, False),
    ([5, 2], [2000, 1500], 700, False), ([130], [0], None, True), ([9], [511], None, False)])
def test_keys_split_over_workgroups(monkeypatch, dtype, d, new, pre, win, sinks):
    # few new tokens over long prefixes: ranges of keys per workgroup, some empty for the shorter
    # requests, merged; and the same call without a workspace that it can use, unsplit
    print(f"[case] extend split {dtype} d={d} new={new} pre={pre} win={win}", flush=True)
    fb, layer, pool, qkv = _batch(new, pre, 8, 2, d, dtype, seed=12, win=win)
    q, k, v = (t.contiguous() for t in qkv.split([8, 2, 2], dim=1))
    kw = {"sinks": torch.randn(8, device=DEV)} if sinks else {}
    got, want = _both(monkeypatch, fb, layer, q, k, v, **kw)
    _close(got, want)
    rows = fb.req_pool_indices.tolist()
    outs = [_direct(q, pool.k_buffer[0], pool.v_buffer[0], fb.req_to_token_pool.req_to_token, rows,
                    new, pre, w, win, kw.get("sinks"))
            for w in (True, False, "short", "unaligned")]
    splits = outs[0][1] > 0
    assert splits == (new != [130])           # 130 keys are too few to split
    for out, _ in outs:
        _close(out.view_as(want), want)
    assert torch.equal(outs[0][0].view_as(got), got)
    assert all(torch.equal(out, outs[1][0]) for out, _ in outs[2 if splits else 0:])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("new,pre,at,nats", [(40, 90, 0, 14), (40, 90, 70, 18), (130, 4000, 0, 16),
                                             (130, 4000, 0, 18), (33, 8000, 4100, 18),
                                             (33, 8000, 0, 24), (33, 8000, 0, 60)])
def test_a_key_that_draws_most_of_the_weight(dtype, d, new, pre, at, nats):
    # a key `nats` above the others whose V is zero: the output is what the small weights sum
    # to. Against float64 the error may be that of rounding the output once, 1 % more at most:
    # beside a rounding of 2e-4 that is an error of the weights below 3e-5 (at 24 nats the
    # outputs are fp16 subnormals, whose rounding is larger; at 60 they are zero)
    print(f"[case] extend peaked {dtype} d={d} new={new} pre={pre} at={at} nats={nats}", flush=True)
    hq, hkv, n = 8, 2, new + pre
    g = torch.Generator(device=DEV).manual_seed(21)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    q, kp, vp = rnd(new, hq, d), rnd(n + 16, hkv, d), 64 + 4 * rnd(n + 16, hkv, d)
    r2t = torch.randperm(n + 16, generator=g, device=DEV)[:n].int()[None]
    q[..., 0], kp[..., 0] = 8.0, 0.0
    kp[r2t[0, at].long(), :, 0] = nats * d ** 0.5 / 8.0
    vp[r2t[0, at].long()] = 0.0
    q, kp, vp = q.to(dtype), kp.to(dtype), vp.to(dtype)
    kk, vv = kp[r2t[0].long()].double(), vp[r2t[0].long()].double()
    mask = torch.arange(n, device=DEV)[None] > torch.arange(pre, n, device=DEV)[:, None]
    want = torch.stack([
        torch.softmax((q[:, i].double() @ kk[:, i // 4].T.contiguous() * d ** -0.5).masked_fill(
            mask, -math.inf), -1) @ vv[:, i // 4] for i in range(hq)], 1)
    rounding = float((want.to(dtype).double() - want).norm())
    for workspace in (True, False):
        got, need = _direct(q, kp, vp, r2t, [0], [new], [pre], workspace)
        assert (need > 0) == (n >= 512)                        # both ways of the kernel
        err = float((got.double() - want).norm())
        assert err <= 1.01 * rounding, (workspace, err / float(want.norm()), rounding / float(want.norm()))


@pytest.mark.gpu
def test_slots_and_rows_count_from_the_end(monkeypatch):
    # negative slots and rows index as PyTorch does; pools as strided views of one buffer
    fb, layer, pool, qkv = _batch([20, 9], [30, 0], 8, 2, 128, torch.float16, seed=8)
    kv = torch.stack([pool.k_buffer[0], pool.v_buffer[0]], dim=1)
    pool.k_buffer[0], pool.v_buffer[0] = kv[:, 0], kv[:, 1]
    r2t = fb.req_to_token_pool.req_to_token
    slots = kv.shape[0]
    r2t.copy_(torch.where(torch.arange(r2t.shape[1], device=DEV) % 2 == 0, r2t - slots, r2t))
    fb.req_pool_indices -= r2t.shape[0]
    q, k, v = (t.contiguous() for t in qkv.split([8, 2, 2], dim=1))
    _close(*_both(monkeypatch, fb, layer, q, k, v))


@pytest.mark.gpu
def test_a_slot_outside_the_pool_gives_nan_to_those_that_see_it():
    fb, layer, pool, qkv = _batch([100], [0], 4, 1, 64, torch.float16, seed=9)
    q, k, v = (t.contiguous() for t in qkv.split([4, 1, 1], dim=1))
    backend = sglang_backend.SplitKVHipBackend()
    backend.forward_extend(q, k, v, layer, fb)
    fb.req_to_token_pool.req_to_token[int(fb.req_pool_indices[0]), 60] = pool.k_buffer[0].shape[0]
    out = backend.forward_extend(q, None, None, layer, fb).view(100, -1)
    assert bool(out[60:].isnan().all()) and not bool(out[:60].isnan().any())


@pytest.mark.gpu
def test_calls_left_to_pytorch(monkeypatch):
    # rows that are not 16-byte aligned, and gradients
    fb, layer, pool, qkv = _batch([5], [4], 4, 2, 64, torch.float16, seed=10)
    q, k, v = (t.contiguous() for t in qkv.split([4, 2, 2], dim=1))
    backend = sglang_backend.SplitKVHipBackend()
    with monkeypatch.context() as m:
        m.setattr(extend, "extend_attention", lambda *a, **b: pytest.fail("kernel path"))
        odd = torch.empty(q.numel() + 1, dtype=q.dtype, device=DEV)[1:].view_as(q).copy_(q)
        want = backend.forward_extend(odd, k, v, layer, fb)
        leaf = q.clone().requires_grad_()
        backend.forward_extend(leaf, k, v, layer, fb).float().sum().backward()
        assert leaf.grad is not None
    _close(backend.forward_extend(q, k, v, layer, fb), want)


@pytest.mark.gpu
def test_a_traced_call_records_its_attention():
    # a call under torch.jit.trace stays on PyTorch, so that the trace computes new inputs
    fb, layer, pool, qkv = _batch([5, 2], [40, 0], 4, 2, 64, torch.float16, seed=14)
    pool.get_key_buffer, pool.get_value_buffer = pool.k_buffer.__getitem__, pool.v_buffer.__getitem__
    backend = sglang_backend.SplitKVHipBackend()
    call = lambda q: backend.forward_extend(q, None, None, layer, fb)  # noqa: E731
    q = qkv[:, :4].contiguous()
    traced = torch.jit.trace(call, (q,), check_trace=False)
    other = q.flip(0).contiguous()
    _close(traced(other), call(other))


def test_what_passes_tensors_through_a_trace_is_not_plain():
    t = torch.zeros(2, 4, 64, dtype=torch.float16)
    seen = []
    torch.jit.trace(lambda x: (seen.append(extend._plain(x)), x + 1)[1], (t,), check_trace=False)
    assert seen == [False] and extend._plain(t)


def test_host_tensors_stay_on_pytorch():
    fb, layer, pool, qkv = _batch([5, 2], [4, 0], 4, 2, 64, torch.float16, seed=11, device="cpu")
    q, k, v = (t.contiguous() for t in qkv.split([4, 2, 2], dim=1))
    out = sglang_backend.SplitKVHipBackend().forward_extend(q, k, v, layer, fb)
    assert out.shape == (7, 4 * 64) and bool(out.isfinite().all())
    r2t = fb.req_to_token_pool.req_to_token
    assert not extend.takes(q, pool.get_key_buffer(0), pool.get_value_buffer(0), r2t, [0], [5],
                            [9], 0.1, None, 1.0, 1.0, None)


def test_split_follows_the_sizes():
    # bytes of (O, m, l) rows: tokens * heads * split * (d + 2) floats
    def split(new, alls, hq=32, hkv=8, d=128, win=0):
        ints = ctypes.c_int32 * len(new)
        b = dk_lib.load().dk_extend_workspace_bytes(len(new), ints(*new), ints(*alls), hq, hkv, d,
                                                    win)
        return b / (4 * sum(new) * hq * (d + 2)) if b else 1

    assert split([2048], [8192]) == 1                     # fills the chip by itself
    assert split([16], [200]) == 1                        # too few keys
    assert 31 < split([16], [8192]) < 33 and 15 < split([64], [4096]) < 17
    assert 1.9 < split([16], [8192], win=512) < 2.1       # bounded by the window
    assert split([0], [100]) == 1


def test_argument_checks():
    # refused before any device call, so without a GPU
    lib = dk_lib.load()

    def call(rows=(0,), new=(2,), alls=(4,), hq=4, hkv=2, d=64, tokens=2, k_s=128, scale=0.1,
             dtype=0, ptr=256, window=0, num_rows=2, stride=8):
        ints = ctypes.c_int32 * len(rows)
        s = dk_lib.DkExtendStrides(hq * d, d, k_s, d, k_s, d, hq * d, d)
        return lib.dk_extend_attention(ptr, ptr, ptr, ptr, stride, num_rows, ints(*rows),
                                       ints(*new), ints(*alls), ptr, None, 0, len(rows), tokens, hq, hkv,
                                       d, 16, dtype, 0, ctypes.byref(s), scale, 1.0, 0.0, window,
                                       None, None)

    assert call(new=(0,)) == 0                                # nothing to do
    for bad in (dict(rows=(2,)), dict(rows=(-1,)), dict(new=(5,)), dict(new=(-1,)),
                dict(alls=(9,)), dict(tokens=1), dict(hq=5), dict(d=96), dict(dtype=7),
                dict(scale=0.0), dict(scale=math.nan), dict(window=-1), dict(k_s=-128)):
        assert call(**bad) < 0, bad
    assert call(k_s=132) == dk_lib.DK_EUNSUPPORTED
    assert call(ptr=8) == dk_lib.DK_EUNSUPPORTED
    assert call(ptr=None) == dk_lib.DK_ENULL
    assert call(new=(0,)) == 0                                # leaves no message behind
