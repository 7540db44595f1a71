"""The native host path (kvq_decode_amd/csrc/host.cpp) against the Python path.

The two must take the same calls with the same results and leave the same errors: the
native functions return None for what they do not take, and the Python path then answers."""
import ctypes
import math

import numpy as np
import pytest
import torch

from kvq_decode_amd import _lib, paged_decode_attention
from kvq_decode_amd.ops import KvqArgumentError


class _Declines:
    """A host module that takes no call."""
    @staticmethod
    def decode(*args):
        return None

    quantize = quantize_append = append_kv = reshape_and_cache = set_cu_count = decode


class _Counts:
    """The host module, counting the calls it takes."""
    def __init__(self, host):
        self.host, self.taken = host, 0

    def __getattr__(self, name):
        f = getattr(self.host, name)

        def call(*args):
            r = f(*args)
            self.taken += r is not None
            return r
        return call


def test_host_declines_what_it_cannot_take():
    """Without a GPU: CPU tensors, other types and wrong argument counts are not taken."""
    assert _lib.HOST_BUILT
    _lib.lib()  # binds the library's functions
    t = torch.zeros(1, 8, 64, dtype=torch.float16)
    for args in ((), (1, 2, 3), (t,) * 18, (None,) * 18):
        assert _lib.host.decode(*args) is None
    for name, n in (("quantize", 5), ("quantize_append", 6), ("append_kv", 6),
                    ("reshape_and_cache", 5)):
        for args in ((), (t,) * n, (None,) * n, ((t,) * 8,) + (t,) * (n - 1)):
            assert getattr(_lib.host, name)(*args) is None
    with pytest.raises(TypeError):
        _lib.host.bind(1)
    with pytest.raises(KvqArgumentError):  # the Python path reports the error
        paged_decode_attention(t, t[None], t[None], t, t)


def _caches(lens, bs, hq, hkv, d, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    pages = [-(-n // bs) for n in lens]
    nb = sum(pages) + 3
    k = torch.randn(nb, bs, hkv, d, generator=g, device="cuda").half()
    v = torch.randn(nb, bs, hkv, d, generator=g, device="cuda").half()
    q = torch.randn(len(lens), hq, d, generator=g, device="cuda").half()
    bt = torch.zeros(len(lens), max(pages) + 1, dtype=torch.int32, device="cuda")
    perm, at = torch.randperm(nb, generator=g, device="cuda").int(), 0
    for b, n in enumerate(pages):
        bt[b, :n] = perm[at:at + n]
        at += n
    return q, k, v, bt, torch.tensor(lens, dtype=torch.int32, device="cuda")


def _both(monkeypatch, call):
    """(result with the native path, calls it took, result with the Python path)."""
    counts = _Counts(_lib.host)
    with monkeypatch.context() as m:
        m.setattr(_lib, "host", counts)
        a = call()
    with monkeypatch.context() as m:
        m.setattr(_lib, "host", _Declines)
        b = call()
    return a, counts.taken, b


@pytest.mark.gpu
@pytest.mark.parametrize("lens", [[700, 3, 129], [4096], [33] * 5])
@pytest.mark.parametrize("fmt", ["fp16", "int8", "int4"])
def test_decode_same_as_python_path(monkeypatch, lens, fmt):
    """The same bits over the forms a call takes; the native path takes all but those that
    need a copy or a conversion."""
    from kvq_decode_amd.quant import quantize_paged_cache
    bs, hq, hkv, d = 16, 8, 2, 64
    q, k, v, bt, sl = _caches(lens, bs, hq, hkv, d)
    kw = {}
    if fmt != "fp16":
        qc = quantize_paged_cache(k, v, bt, sl, fmt)
        k, v, kw = qc.k_codes, qc.v_codes, qc.decode_kwargs()
    B = len(lens)
    wide = torch.randn(B, hq + 4, d, device="cuda").half()
    odd = torch.randn(B, hq, d + 1, device="cuda").half()
    out = torch.empty(B, hq + 1, d, dtype=torch.float16, device="cuda")
    ws = (torch.empty(hq * (64 + B) * d, device="cuda"), torch.empty(hq * (64 + B), device="cuda"))
    forms = [  # (positional after seq_lens, keywords, q, taken)
        ((), {}, q, 1), ((0.3,), {}, q, 1), ((None, 1), {}, q, 1), ((None, 3), {}, q, 1),
        ((), dict(units=7), q, 1), ((), dict(units=5, workspace=ws, waves_per_group=1), q, 1),
        ((None, 2), dict(workspace=ws, out=out[:, :hq]), q, 1), ((), dict(pipeline=1), q, 1),
        ((), {}, wide[:, 2:2 + hq], 1),
        ((), {}, odd[..., :d], 0),                       # rows that are not 16-byte aligned
        ((np.float32(0.3),), {}, q, 0), ((1,), {}, q, 0),  # converted by the Python path
        ((None, np.int64(3)), {}, q, 0), ((), dict(check_seq_lens=True), q, 0)]
    paged_decode_attention(q, k, v, bt, sl, **kw)  # the CU count of the device is known now
    for args, more, qq, taken in forms:
        a, n, b = _both(monkeypatch, lambda: paged_decode_attention(
            qq, k, v, bt, sl, *args, **kw, **more).clone())
        assert n == taken, (args, list(more))
        assert torch.equal(a, b), (args, list(more))
    given = out[:, :hq]
    assert paged_decode_attention(q, k, v, bt, sl, out=given, **kw) is given


@pytest.mark.gpu
def test_errors_same_as_python_path(monkeypatch):
    """Every refused call raises what it raises without the native path."""
    _lib.lib()  # binds the library's functions
    q, k, v, bt, sl = _caches([300, 40], 16, 8, 2, 64)
    ws = (torch.empty(8, device="cuda"), torch.empty(8, device="cuda"))
    bad = [dict(q=q.float()), dict(k_cache=k.float()), dict(v_cache=v[1:]), dict(k_cache=k[..., :32]),
           dict(block_table=bt.long()), dict(seq_lens=sl[:1]), dict(block_table=bt.t()),
           dict(seq_lens=sl.cpu()), dict(q=q[:, :7]), dict(num_splits=2, units=3), dict(units=-1),
           dict(kv_format="int8"), dict(kv_format="none"), dict(out=q[:, :4]), dict(units=4, workspace=ws),
           dict(scale=math.nan), dict(waves_per_group=3), dict(pipeline=7), dict(num_splits=2, workspace=ws),
           dict(k_cache=k[:, :8], v_cache=v[:, :8])]
    for change in bad:
        call = dict(q=q, k_cache=k, v_cache=v, block_table=bt, seq_lens=sl, **{
            n: x for n, x in change.items() if n not in ("q", "k_cache", "v_cache", "block_table", "seq_lens")})
        call.update(change)
        seen = []
        for host in (_lib.host, _Declines):
            with monkeypatch.context() as m:
                m.setattr(_lib, "host", host)
                with pytest.raises((AssertionError, RuntimeError)) as e:
                    paged_decode_attention(**call)
            seen.append((type(e.value), str(e.value)))
        assert seen[0] == seen[1], change


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["int8", "int4"])
def test_write_paths_same_as_python_path(monkeypatch, fmt):
    """Bulk quantizer, quantized append, fp16 append and slot scatter: every byte."""
    from kvq_decode_amd.cache import append_kv, reshape_and_cache
    from kvq_decode_amd.quant import (allocate_quantized_cache, init_k_residual, quantize_append,
                                      quantize_paged_cache)
    _, k, v, bt, sl = _caches([300, 40], 16, 8, 2, 64)
    new = torch.randn(2, 2, 2, 64, device="cuda").half()
    rows = torch.randn(9, 8, 64, device="cuda").half()
    slots = torch.tensor([5, 40, -1, 17, 99, 200, 3, 64, 65], device="cuda")

    def write():
        qc = allocate_quantized_cache(k.shape[0], 16, 2, 64, fmt, "cuda")
        for t in qc[:6]:
            t.zero_()
        quantize_paged_cache(k, v, bt, sl, fmt, out=qc)
        resid = init_k_residual(k, bt, sl)
        quantize_append(qc, new[0], new[1], bt, sl + 1, resid)
        kc, vc = k.clone(), v.clone()
        append_kv(kc, vc, new[0], new[1], bt, sl + 1)
        reshape_and_cache(rows[:, 1:3], rows[:, 5:7], kc, vc, slots)
        return [t.contiguous().view(torch.uint8) for t in (*qc[:6], resid, kc, vc)]

    a, taken, b = _both(monkeypatch, write)
    assert taken == 4
    assert all(torch.equal(x, y) for x, y in zip(a, b))
    for f, args in ((append_kv, (k, v, new[0].float(), new[1], bt, sl)),
                    (append_kv, (k, v, new[0, :1], new[1], bt, sl)),
                    (reshape_and_cache, (rows[:, 1:3], rows[:, 5:7], k, v, slots.int())),
                    (reshape_and_cache, (rows[:, 1:4], rows[:, 5:8], k, v, slots))):
        with pytest.raises(KvqArgumentError):
            f(*args)


@pytest.mark.gpu
def test_launch_error_is_raised_after_one_call():
    """A library function that reports a failed launch is called once and its status raised: a
    second call through the Python path could return normally and hide it. The functions that
    launch are host-side stand-ins here; no kernel runs."""
    from kvq_decode_amd.cache import append_kv, reshape_and_cache
    from kvq_decode_amd.quant import (allocate_quantized_cache, init_k_residual, quantize_append,
                                      quantize_paged_cache)
    q, k, v, bt, sl = _caches([300, 40], 16, 8, 2, 64)
    new, slots = k[0, :2].contiguous(), torch.zeros(2, dtype=torch.int64, device="cuda")
    qc = allocate_quantized_cache(k.shape[0], 16, 2, 64, "int8", "cuda")
    resid = init_k_residual(k, bt, sl)
    paged_decode_attention(q, k, v, bt, sl)  # the CU count of the device is known now
    launches = ("kvq_paged_decode", "kvq_decode_units", "kvq_quantize_cache",
                "kvq_quantize_append", "kvq_append_kv", "kvq_reshape_and_cache")
    calls = []

    class Failing:
        """The library, with every launching function replaced."""
        kept = []

        def __getattr__(self, name):
            f = getattr(_lib.lib(), name)
            if name not in launches:
                return f
            params = [ctypes.c_void_p if t not in (ctypes.c_int32, ctypes.c_int64) else t
                      for t in f.argtypes]
            stub = ctypes.CFUNCTYPE(ctypes.c_int, *params)(
                lambda *a: calls.append(name) or _lib.KVQ_ERR_HIP)
            self.kept.append(stub)
            return stub

    try:
        _lib.bind_host(Failing())
        for name, call in (
                ("kvq_paged_decode", lambda: paged_decode_attention(q, k, v, bt, sl, None, 1)),
                ("kvq_decode_units", lambda: paged_decode_attention(q, k, v, bt, sl, units=3)),
                ("kvq_quantize_cache", lambda: quantize_paged_cache(k, v, bt, sl, "int8", out=qc)),
                ("kvq_quantize_append", lambda: quantize_append(qc, new, new, bt, sl, resid)),
                ("kvq_append_kv", lambda: append_kv(k, v, new, new, bt, sl)),
                ("kvq_reshape_and_cache", lambda: reshape_and_cache(new, new, k, v, slots))):
            calls.clear()
            with pytest.raises(_lib.KvqError) as e:
                call()
            assert calls == [name] and e.value.status == _lib.KVQ_ERR_HIP
    finally:
        _lib.bind_host(_lib.lib())
    assert torch.equal(paged_decode_attention(q, k, v, bt, sl), paged_decode_attention(q, k, v, bt, sl))
