"""Mask preparation (vx_key_masks_fwd, vx_full_bias_fwd): one launch each,
compared bit for bit with the elementwise definition in numpy, over the forms
a mask may come in: expanded, transposed, offset and strided views, widths
around the 16-key vectors and 64-key tiles, one pass of a workgroup and more,
infinities and NaN."""
import ctypes

import numpy as np
import pytest
import torch

from vidax_amd import _lib

A = 1 << 20  # a 16-byte aligned fake device address (never dereferenced)


@pytest.mark.parametrize("kw,frag", [
    (dict(valid=None), "valid or bias"),
    (dict(B=0), ">= 1"),
    (dict(bias_rows=A), "needs its input"),
    (dict(rows=A + 8), "aligned"),
    (dict(stride=250), "row_stride"),
    (dict(stride=192), "row_stride"),
    (dict(strides=(-1, 1)), "strides"),
    (dict(strides=None), "strides"),
])
def test_key_masks_rejects(kw, frag):
    a = dict(valid=A, strides=(200, 1), B=1, Sk=200, rows=A, bias_rows=None, stride=256)
    a.update(kw)
    st = _lib.strides2(a["strides"]) if a["strides"] is not None else None
    rc = _lib.lib().vx_key_masks_fwd(a["valid"], st, None, None, a["B"], a["Sk"], None, a["rows"], a["bias_rows"],
                                     a["stride"], None)
    assert rc == _lib.VX_ERR_INVALID_ARGUMENT and frag in _lib.last_error(), _lib.last_error()


@pytest.mark.parametrize("kw,frag", [
    (dict(bias=None), "bias or mask"),
    (dict(out=A + 4), "aligned"),
    (dict(bias=A + 2), "aligned"),
    (dict(Sk=0), ">= 1"),
    (dict(strides=(0, 0, -64, 1)), "strides"),
])
def test_full_bias_rejects(kw, frag):
    a = dict(bias=A, strides=(0, 0, 64, 1), Sk=64, out=A)
    a.update(kw)
    st = (ctypes.c_int64 * 4)(*a["strides"])
    rc = _lib.lib().vx_full_bias_fwd(a["bias"], st, None, None, 1, 1, 8, a["Sk"], a["out"], None)
    assert rc == _lib.VX_ERR_INVALID_ARGUMENT and frag in _lib.last_error(), _lib.last_error()


def _biases(shape, rng):
    x = rng.standard_normal(shape).astype(np.float32)
    x[rng.random(shape) < 0.3] = -np.inf
    x[rng.random(shape) < 0.05] = np.inf
    x[rng.random(shape) < 0.05] = np.nan
    return x


@pytest.mark.gpu
@pytest.mark.parametrize("Sk", [1, 15, 16, 17, 63, 64, 65, 333, 4096, 16385, 40001])
@pytest.mark.parametrize("form", ["contiguous", "expanded", "transposed", "offset", "strided", "scalar_key"])
def test_key_masks(gpu, Sk, form):
    from vidax_amd.attention import _KeyMasks
    B = 3
    rng = np.random.default_rng(Sk)
    print(f"[case] key masks Sk={Sk} {form}", flush=True)

    def view(x):
        t = torch.from_numpy(x).to(gpu)
        if form == "expanded":
            return t[:1].expand(B, Sk)
        if form == "transposed":
            return t.t().contiguous().t()
        if form == "offset":
            w = torch.zeros((B, Sk + 3), dtype=t.dtype, device=gpu)
            w[:, 3:] = t
            return w[:, 3:]
        if form == "strided":
            w = torch.zeros((B, Sk, 2), dtype=t.dtype, device=gpu)
            w[..., 1] = t
            return w[..., 1]
        if form == "scalar_key":
            return t[:, :1].expand(B, Sk)
        return t

    valid = view(rng.random((B, Sk)) < 0.6)
    bias = view(_biases((B, Sk), rng))
    vn, bn = valid.cpu().numpy(), bias.cpu().numpy()
    for use_v, use_b in ((True, False), (False, True), (True, True)):
        m = _KeyMasks(valid if use_v else None, bias if use_b else None, want_len=True)
        assert _lib.last_launch() == "key_mask_kernel"
        torch.cuda.synchronize()
        buf = m.buf.cpu().numpy()
        ok = (vn if use_v else True) & ((bn > -np.inf) if use_b else True)
        pos = np.where(np.broadcast_to(ok, (B, Sk)), np.arange(1, Sk + 1), 0)
        assert np.array_equal(buf[:4 * B].view(np.int32), pos.max(1))
        if use_b:
            rows = buf[m.bias_off:m.bias_off + 4 * B * m.stride].view(np.uint32).reshape(B, m.stride)
            assert np.array_equal(rows[:, :Sk], np.ascontiguousarray(bn).view(np.uint32))
            assert (rows[:, Sk:] == 0xff800000).all()
        if use_v:
            rows = buf[m.valid_off:].reshape(B, m.stride)
            assert np.array_equal(rows[:, :Sk], vn.astype(np.uint8)) and (rows[:, Sk:] == 0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("Sk,Sq", [(1, 5), (3, 5), (64, 5), (77, 5), (257, 5), (512, 5), (1, 64), (504, 130),
                                   (505, 130), (1024, 64), (1023, 65), (4161, 70)])
@pytest.mark.parametrize("bias_shape,mask_shape", [
    (None, (1, 1, 5, 0)), ((1, 3, 5, 0), None), ((1, 3, 5, 0), (2, 1, 5, 0)), ((2, 3, 1, 0), (1, 1, 5, 0)),
    ((2, 1, 5, 1), (5, 0)), ((3, 5, 0), (2, 1, 1, 1)), ((1, 3, 5, 1), None), ((2, 3, 5, 0), None), ((5, 1), None),
    ((1, 1, 1, 0), None),
])
def test_full_bias(gpu, Sk, Sq, bias_shape, mask_shape):
    """A 0 extent stands for Sk, a 5 for Sq. Inputs of 65536 scores a head
    and more with the key dim strided and the queries next to each other go
    through 64 x 64 tiles."""
    from vidax_amd.attention import _full_bias
    B, H = 2, 3
    rng = np.random.default_rng(Sk)
    shape = lambda s: tuple({0: Sk, 5: Sq}.get(n, n) for n in s)
    print(f"[case] full bias Sk={Sk} Sq={Sq} bias={bias_shape} mask={mask_shape}", flush=True)
    bias = _biases(shape(bias_shape), rng) if bias_shape else None
    mask = rng.random(shape(mask_shape)) < 0.5 if mask_shape else None
    ref = np.zeros((B, H, Sq, Sk), np.float32)
    if bias is not None:
        ref = ref + bias
    if mask is not None:
        with np.errstate(invalid="ignore"):
            ref = ref + np.where(mask, np.float32(0), np.float32(-np.inf))
    for transposed in (False, True):
        t = lambda x: None if x is None else torch.from_numpy(x).to(gpu)
        tb, tm = t(bias), t(mask)
        if transposed:  # the key dim strided
            tb = None if tb is None else tb.transpose(-1, -2).contiguous().transpose(-1, -2)
            tm = None if tm is None else tm.transpose(-1, -2).contiguous().transpose(-1, -2)
        x, st = _full_bias(tb, B, H, Sq, Sk, gpu, tm)
        if x is not tb:
            lead = tb if tb is not None else tm
            qs, ks = [0 if n == 1 else s for n, s in zip(lead.shape, lead.stride())][-2:]
            tiles = 0 < qs < ks and max(y.shape[-2] for y in (tb, tm) if y is not None) * Sk >= 65536
            want = "full_bias_transposed_kernel" if tiles else "full_bias_kernel"
            assert _lib.last_launch() == want, (_lib.last_launch(), qs, ks)
        got = torch.as_strided(x, (B, H, Sq, Sk), (*st, 1)).cpu().numpy()
        assert x.data_ptr() % 16 == 0 and all(s % 4 == 0 for s in st)
        assert np.array_equal(got, ref, equal_nan=True)
        assert np.array_equal(np.signbit(got) & ~np.isnan(ref), np.signbit(ref) & ~np.isnan(ref))


@pytest.mark.gpu
def test_masked_calls_under_graph_capture(gpu):
    """The mask launches are captured with the call: every replay follows the
    masks' contents."""
    from vidax_amd import dot_product_attention, masked_self_attention
    g = torch.Generator(device=gpu).manual_seed(5)
    q, k, v = (torch.randn((2, 150, 2, 64), generator=g, device=gpu).to(torch.bfloat16) for _ in range(3))
    valid = torch.ones((2, 150), dtype=torch.bool, device=gpu)
    causal = torch.ones((150, 150), dtype=torch.bool, device=gpu).tril()[None, None].contiguous()
    run = lambda: (masked_self_attention(q, k, v, key_valid=valid), dot_product_attention(q, k, v, mask=causal))
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = run()
    for step in range(3):
        valid[:, 100 - 20 * step:] = False
        causal[..., step::7] = step == 1
        causal[..., 0] = True
        eager = run()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(outs, eager):
            assert torch.equal(a, b), step


@pytest.mark.gpu
@pytest.mark.parametrize("Sk", [2 ** 31 - 100, 2 ** 31 - 1])
def test_masks_of_the_longest_rows(gpu, Sk):
    """seq_k up to 2^31 - 1: the key counters run past 2^31 (round_up(seq_k,
    64) and the step behind the last pass), so they are 64-bit. The inputs are
    one element read at key stride 0."""
    print(f"[case] mask rows of {Sk} keys", flush=True)
    L = _lib.lib()
    width = (Sk + 63) // 64 * 64
    stream = torch.cuda.current_stream().cuda_stream
    one = torch.ones(1, dtype=torch.uint8, device=gpu)
    rows = torch.full((width,), 7, dtype=torch.uint8, device=gpu)
    kv_len = torch.zeros(1, dtype=torch.int32, device=gpu)
    _lib.raise_for(L.vx_key_masks_fwd(one.data_ptr(), _lib.strides2((0, 0)), None, None, 1, Sk, kv_len.data_ptr(),
                                      rows.data_ptr(), None, width, stream))
    torch.cuda.synchronize()
    assert kv_len.item() == Sk
    assert (rows[:Sk] == 1).all() and (rows[Sk:] == 0).all()
    del rows
    bias = torch.full((1,), 2.5, device=gpu)
    out = torch.full((width,), 7.0, device=gpu)
    zero = (ctypes.c_int64 * 4)(0, 0, 0, 0)
    _lib.raise_for(L.vx_full_bias_fwd(bias.data_ptr(), zero, None, None, 1, 1, 1, Sk, out.data_ptr(), stream))
    torch.cuda.synchronize()
    assert (out[:Sk] == 2.5).all() and (out[Sk:] == 0).all()


def _neg_view(x):
    """x's values in a view whose memory holds them negated (the imaginary
    part of a conjugate, as torch gives it)."""
    y = torch.complex(torch.zeros_like(x), -x).conj().imag
    assert y.is_neg() and torch.equal(y, x)
    return y


def test_as_dtype_resolves_negated_views():
    x = torch.arange(6.0).reshape(2, 3)
    y = _lib.as_dtype(_neg_view(x), x.device, torch.float32)
    assert not y.is_neg() and torch.equal(y, x)
    assert _lib.as_dtype(x, x.device, torch.float32) is x


@pytest.mark.gpu
def test_negated_views(gpu):
    """Biases, norm weights and rope tables given as views that torch marks as
    negated count with their values, not with what their memory holds."""
    from vidax_amd import (create_abs_rope3d_freqs, dot_product_attention, flash_attention, na3d_qk_norm_rope,
                           rms_norm)
    print("[case] negated views", flush=True)
    g = torch.Generator(device=gpu).manual_seed(6)
    q, k, v = (torch.randn((1, 64, 2, 64), generator=g, device=gpu).to(torch.bfloat16) for _ in range(3))
    kb = torch.randn((1, 1, 1, 64), generator=g, device=gpu)
    fb = torch.randn((1, 2, 64, 64), generator=g, device=gpu)
    for b in (kb, fb, fb[:, :, :, :1]):
        assert torch.equal(dot_product_attention(q, k, v, bias=_neg_view(b)), dot_product_attention(q, k, v, bias=b))
    assert torch.equal(flash_attention(q, k, v, key_bias=_neg_view(kb).reshape(1, 64)),
                       flash_attention(q, k, v, key_bias=kb.reshape(1, 64)))
    x = torch.randn((1, 2, 3, 5, 3, 64), generator=g, device=gpu).to(torch.bfloat16)
    w = torch.randn(64, generator=g, device=gpu)
    freqs = create_abs_rope3d_freqs(2, 3, 5, 64, device=gpu)
    assert torch.equal(na3d_qk_norm_rope(x, _neg_view(w), tuple(_neg_view(t) for t in freqs)),
                       na3d_qk_norm_rope(x, w, freqs))
    y = x.reshape(1, -1, 3, 64)
    assert torch.equal(rms_norm(y, _neg_view(w)), rms_norm(y, w))
