"""GPU parity tests of the flash-attention kernel against the CPU oracle.

Bar (from the path's specification): max-abs <= 2e-2 and mean-abs <= 2e-3
against the reference semantics, bf16 in/out with fp32 softmax statistics.
Each test also checks the error relative to the output RMS, which catches
mistakes that the absolute bound alone would let through on tiny outputs.
"""
import math
import re

import numpy as np
import pytest
import torch

from oracle import attention_oracle as O

pytestmark = pytest.mark.gpu

MAX_ABS = 2e-2
MEAN_ABS = 2e-3
MEAN_REL_RMS = 1e-2  # mean-abs error / RMS(reference)


def _say(msg):
    print(f"[case] {msg}", flush=True)


def _t(x, dev):
    return torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).to(dev).to(torch.bfloat16)


def _errs(out, ref):
    o = out.float().cpu().numpy().astype(np.float64)
    d = np.abs(o - ref)
    rms = float(np.sqrt(np.mean(ref ** 2))) + 1e-30
    return float(d.max()), float(d.mean()), float(d.mean()) / rms


def _check(out, ref, label):
    mx, mean, rel = _errs(out, ref)
    print(f"  {label}: max_abs={mx:.3e} mean_abs={mean:.3e} mean/rms={rel:.3e}", flush=True)
    assert np.isfinite(out.float().cpu().numpy()).all(), f"{label}: non-finite output"
    assert mx <= MAX_ABS, f"{label}: max-abs {mx}"
    assert mean <= MEAN_ABS, f"{label}: mean-abs {mean}"
    assert rel <= MEAN_REL_RMS, f"{label}: mean-abs/rms {rel}"


SMALL_CASES = [
    # B, Sq, Sk, H, seed, mask
    (1, 128, 128, 2, 10, None),
    (1, 64, 64, 1, 11, None),
    (2, 200, 300, 3, 12, None),          # ragged query and key tails
    (1, 1, 1, 1, 13, None),
    (1, 257, 1, 2, 14, None),            # Sk = 1: out = v
    (1, 33, 65, 2, 15, None),
    (1, 300, 1000, 2, 16, None),         # several key tiles + tail 40
    (3, 100, 777, 2, 17, ("kv_len", 0, 777)),
    (2, 130, 512, 4, 18, ("kv_len", 20, 512)),   # the cross-attention regime
    (2, 96, 515, 2, 19, ("tail_pad", 0, 200)),   # joint text+video padding
]


@pytest.mark.parametrize("B,Sq,Sk,H,seed,mask", SMALL_CASES)
def test_flash_small(gpu, B, Sq, Sk, H, seed, mask):
    from vidax_amd import flash_attention
    _say(f"flash small B={B} Sq={Sq} Sk={Sk} H={H} seed={seed} mask={mask}")
    q, k, v, extra = O.make_flash_inputs(B, Sq, Sk, H, 128, seed, mask)
    kw = {}
    if "kv_len" in extra:
        kw["kv_len"] = torch.from_numpy(extra["kv_len"]).to(gpu)
    if "key_valid" in extra:
        kw["key_valid"] = torch.from_numpy(extra["key_valid"]).to(gpu)
    out = flash_attention(_t(q, gpu), _t(k, gpu), _t(v, gpu), **kw)
    torch.cuda.synchronize()
    ref = O.attention(q, k, v, kv_len=extra.get("kv_len"), key_valid=extra.get("key_valid"))
    _check(out, ref, "oracle")


@pytest.mark.parametrize("B,Sq,Sk,H,D,scale,seed", [
    (1, 300, 777, 3, 128, None, 20),     # default scale 1/sqrt(D)
    (2, 200, 129, 2, 64, 0.3, 21),       # explicit scale, head dim 64
    (1, 2048, 2048, 8, 128, 1.0, 22),    # scale 1
])
def test_local_attention(gpu, B, Sq, Sk, H, D, scale, seed):
    """local_attention (`src/vidax/core/attention.py:321-338`): the unmasked
    kernel with the reference's scale rule (1/sqrt(D) unless given)."""
    from vidax_amd import _lib, local_attention
    _say(f"local_attention B={B} Sq={Sq} Sk={Sk} H={H} D={D} scale={scale}")
    q, k, v, _ = O.make_flash_inputs(B, Sq, Sk, H, D, seed)
    out = local_attention(_t(q, gpu), _t(k, gpu), _t(v, gpu), scale=scale)
    torch.cuda.synchronize()
    assert re.fullmatch(r"flash_(fwd|pair)_(split_)?kernel<0, .*>", _lib.last_launch()), _lib.last_launch()
    assert out.shape == (B, Sq, H, D) and out.dtype == torch.bfloat16
    ref = O.attention(q, k, v, scale=D ** -0.5 if scale is None else scale)
    _check(out, ref, "oracle")


ROW_SHIFTS = [-1000.0, -120.0, 200.0, 1000.0]


@pytest.mark.parametrize("shift", ROW_SHIFTS)
@pytest.mark.parametrize("masked", [False, True])
def test_flash_row_offsets(gpu, shift, masked):
    """A constant added to every score of a query row leaves its softmax
    unchanged. Key dim 0 is all ones and the query's dim 0 is `shift` (every
    other query row 0), scale 1: rows whose scores all lie far below 2^-100
    or far above 2^8 (log2 units) next to ordinary rows in the same wave
    must still match the oracle, which subtracts each row's max."""
    from vidax_amd import flash_attention
    _say(f"flash row offsets shift={shift} masked={masked}")
    B, Sq, Sk, H, D = 2, 96, 300, 2, 128
    rng = np.random.default_rng(70)
    q = O.bf16_round((0.3 * rng.standard_normal((B, Sq, H, D))).astype(np.float32))
    k = O.bf16_round((0.3 * rng.standard_normal((B, Sk, H, D))).astype(np.float32))
    v = O.bf16_round(rng.standard_normal((B, Sk, H, D)).astype(np.float32))
    k[..., 0] = 1.0
    q[:, ::2, :, 0] = shift
    q[:, 1::2, :, 0] = 0.0
    kv_len = np.array([Sk, 170], np.int32) if masked else None
    out = flash_attention(_t(q, gpu), _t(k, gpu), _t(v, gpu), scale=1.0,
                          kv_len=torch.from_numpy(kv_len).to(gpu) if masked else None)
    torch.cuda.synchronize()
    _check(out, O.attention(q, k, v, scale=1.0, kv_len=kv_len), "oracle")


def test_flash_sk1_returns_v(gpu):
    """Sk = 1: every query attends one key with weight 1, so out = v."""
    from vidax_amd import flash_attention
    _say("flash Sk=1 identity")
    q, k, v, _ = O.make_flash_inputs(2, 70, 1, 3, 128, 20)
    out = flash_attention(_t(q, gpu), _t(k, gpu), _t(v, gpu)).float().cpu().numpy()
    np.testing.assert_array_equal(out, np.broadcast_to(v, out.shape))


def test_flash_fully_masked_rows_are_zero(gpu):
    from vidax_amd import flash_attention
    _say("flash fully masked batch item")
    q, k, v, _ = O.make_flash_inputs(2, 50, 130, 2, 128, 21)
    kv_len = torch.tensor([0, 130], dtype=torch.int32, device=gpu)
    out = flash_attention(_t(q, gpu), _t(k, gpu), _t(v, gpu), kv_len=kv_len)
    o = out.float().cpu().numpy()
    assert (o[0] == 0).all()
    ref = O.attention(q[1:], k[1:], v[1:])
    _check(out[1:], ref, "unmasked item")


def test_flash_general_key_mask_and_bias(gpu):
    """key_valid with holes and an additive key bias with -inf entries."""
    from vidax_amd import flash_attention
    _say("flash key_valid holes + key_bias")
    rng = np.random.default_rng(22)
    B, Sq, Sk, H = 2, 150, 333, 2
    q, k, v, _ = O.make_flash_inputs(B, Sq, Sk, H, 128, 22)
    valid = rng.random((B, Sk)) > 0.3
    bias = rng.standard_normal((B, Sk)).astype(np.float32)
    bias[rng.random((B, Sk)) < 0.1] = -np.inf
    tq, tk, tv = _t(q, gpu), _t(k, gpu), _t(v, gpu)
    out = flash_attention(tq, tk, tv, key_valid=torch.from_numpy(valid).to(gpu))
    _check(out, O.attention(q, k, v, key_valid=valid), "key_valid")
    out = flash_attention(tq, tk, tv, key_bias=torch.from_numpy(bias).to(gpu))
    _check(out, O.attention(q, k, v, key_bias=bias), "key_bias")
    kv_len = np.array([100, 333], dtype=np.int32)
    out = flash_attention(tq, tk, tv, key_valid=torch.from_numpy(valid).to(gpu),
                          key_bias=torch.from_numpy(bias).to(gpu),
                          kv_len=torch.from_numpy(kv_len).to(gpu))
    _check(out, O.attention(q, k, v, key_valid=valid, key_bias=bias, kv_len=kv_len), "all three")


def test_flash_scale_and_strided_views(gpu):
    """scale = 1.0 (T5 convention) and q/k/v taken as views of a fused qkv tensor."""
    from vidax_amd import flash_attention
    _say("flash scale=1 strided views")
    B, S, H, D = 2, 190, 3, 128
    rng = np.random.default_rng(23)
    qkv = O.bf16_round(rng.standard_normal((B, S, 3, H, D), dtype=np.float32) * np.float32(0.2))
    t = _t(qkv, gpu)
    q, k, v = t[:, :, 0], t[:, :, 1], t[:, :, 2]
    assert not q.is_contiguous()
    out = flash_attention(q, k, v, scale=1.0)
    ref = O.attention(qkv[:, :, 0], qkv[:, :, 1], qkv[:, :, 2], scale=1.0)
    _check(out, ref, "strided")
    out2 = flash_attention(q.contiguous(), k.contiguous(), v.contiguous(), scale=1.0)
    assert torch.equal(out, out2)


def test_flash_deterministic(gpu):
    from vidax_amd import flash_attention
    _say("flash determinism")
    q, k, v, _ = O.make_flash_inputs(1, 500, 700, 4, 128, 24)
    tq, tk, tv = _t(q, gpu), _t(k, gpu), _t(v, gpu)
    a = flash_attention(tq, tk, tv)
    b = flash_attention(tq, tk, tv)
    assert torch.equal(a, b)


def test_flash_config1_full(gpu):
    """Wan2.1-1.3B self-attention, B=1 H=12 L=7800 D=128, seed 0, whole output."""
    from vidax_amd import flash_attention
    _say("flash c1 full B=1 H=12 L=7800")
    from vidax_amd import _lib
    q, k, v, _ = O.make_flash_inputs(1, 7800, 7800, 12, 128, 0)
    out = flash_attention(_t(q, gpu), _t(k, gpu), _t(v, gpu))
    # 732 workgroups for 512 resident ones: the last 220 run split over the key halves
    assert _lib.last_launch() == "flash_fwd_split_kernel<0, 128, 4>", _lib.last_launch()
    ref = O.attention(q, k, v, acc=np.float32)
    _check(out, ref, "c1")


def _residue_rows(n_total, per_residue, seed):
    """Query rows covering every position of a 256-query workgroup tile
    (every residue mod 256: all 8 waves x 32 query lanes) `per_residue` times,
    in tiles spread over the sequence, plus the first and last rows."""
    rng = np.random.default_rng(seed)
    rows = {0, n_total - 1}
    for r in range(256):
        tiles = np.arange((n_total - 1 - r) // 256 + 1)
        rows.update(int(r + 256 * t) for t in rng.choice(tiles, size=min(per_residue, len(tiles)), replace=False))
    return np.array(sorted(rows))


def _rows(n_total, n, seed):
    rng = np.random.default_rng(seed)
    rows = rng.choice(n_total, size=n, replace=False)
    rows[:2] = [0, n_total - 1]
    return np.sort(rows)


def _torch_inputs(B, Sq, Sk, H, seed, dev):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    q = torch.randn((B, Sq, H, 128), generator=g, device=dev, dtype=torch.float32).to(torch.bfloat16)
    k = torch.randn((B, Sk, H, 128), generator=g, device=dev, dtype=torch.float32).to(torch.bfloat16)
    v = torch.randn((B, Sk, H, 128), generator=g, device=dev, dtype=torch.float32).to(torch.bfloat16)
    return q, k, v


def _np(t):
    return t.float().cpu().numpy()


@pytest.mark.slow
def test_flash_config2_sampled_rows(gpu):
    """Headline shape B=1 H=40 L=32760: 514 sampled query rows (all heads)
    vs the oracle, two per position of a 256-query workgroup tile."""
    from vidax_amd import _lib, flash_attention
    _say("flash c2 B=1 H=40 L=32760 sampled rows")
    q, k, v = _torch_inputs(1, 32760, 32760, 40, 1, gpu)
    out = flash_attention(q, k, v)
    assert _lib.last_launch() == "flash_fwd_kernel<0, 128, 8>", _lib.last_launch()
    rows = _residue_rows(32760, 2, 1)
    assert len(rows) >= 512
    ref = O.attention_rows(_np(q), _np(k), _np(v), rows)
    _check(out[:, torch.from_numpy(rows).to(gpu)], ref, "c2 rows")


@pytest.mark.slow
def test_flash_config3_cross_kvlen(gpu):
    """Cross attention Lq=32760, Lk=512, B=2 H=40, kv_len ~ U{20..512}."""
    from vidax_amd import flash_attention
    _say("flash c3 cross B=2 H=40 Lq=32760 Lk=512 kv_len")
    q, k, v = _torch_inputs(2, 32760, 512, 40, 2, gpu)
    kv_len = np.random.default_rng(2).integers(20, 513, size=2).astype(np.int32)
    from vidax_amd import _lib
    out = flash_attention(q, k, v, kv_len=torch.from_numpy(kv_len).to(gpu))
    assert _lib.last_launch() == "flash_stream_kernel<128>", _lib.last_launch()
    rows = _rows(32760, 512, 2)
    ref = O.attention_rows(_np(q), _np(k), _np(v), rows, kv_len=kv_len)
    _check(out[:, torch.from_numpy(rows).to(gpu)], ref, "c3 rows")
    # the same mask as a boolean key mask through dot_product_attention
    from vidax_amd import dot_product_attention
    valid = torch.arange(512, device=gpu)[None, :] < torch.from_numpy(kv_len).to(gpu)[:, None]
    out2 = dot_product_attention(q, k, v, mask=valid[:, None, None, :])
    assert torch.equal(out, out2)


@pytest.mark.slow
def test_flash_config5_joint_sampled_rows(gpu):
    """Joint text+video B=1 H=24, S = 33*45*80 + 256 = 119056, last p ~ U{0..200}
    keys invalid; 514 sampled query rows, two per position of a 256-query tile."""
    from vidax_amd import masked_self_attention
    _say("flash c5 joint B=1 H=24 S=119056 key padding")
    S = 33 * 45 * 80 + 256
    q, k, v = _torch_inputs(1, S, S, 24, 4, gpu)
    p = int(np.random.default_rng(4).integers(0, 201))
    valid = torch.ones((1, S), dtype=torch.bool, device=gpu)
    if p:
        valid[:, S - p:] = False
    out = masked_self_attention(q, k, v, key_valid=valid).reshape(1, S, 24, 128)
    from vidax_amd import _lib, flash_attention
    # the key-validity kernel (its tiles classified on the device: all but
    # the tail tile take the unmasked path)
    assert _lib.last_launch() == "flash_fwd_kernel<1, 128, 8>", _lib.last_launch()
    # the same mask as kv_len alone: the unmasked kernel, at full size
    kv_len = valid.to(torch.int32).sum(dim=1, dtype=torch.int32)
    out_kvlen = flash_attention(q, k, v, scale=128 ** -0.5, kv_len=kv_len)
    assert _lib.last_launch() == "flash_fwd_kernel<0, 128, 8>", _lib.last_launch()
    d = (out.float() - out_kvlen.float()).abs()
    assert d.max().item() <= 1e-2 and d.mean().item() <= 1e-4, (d.max().item(), d.mean().item())
    del out_kvlen, d
    rows = _residue_rows(S, 2, 4)
    assert len(rows) >= 512
    ref = O.attention_rows(_np(q), _np(k), _np(v), rows, key_valid=_np(valid).astype(bool))
    _check(out[:, torch.from_numpy(rows).to(gpu)], ref, f"c5 rows (p={p})")


@pytest.mark.slow
def test_flash_config5_zero_query_is_valid_mean(gpu):
    """Full-size invariant: q = 0 gives uniform weights, so every output row is
    the mean of the valid V rows (pins masking, accumulation over all 119k
    keys and the normalisation, independently of the oracle)."""
    from vidax_amd import flash_attention
    _say("flash c5 q=0 mean-of-valid-V invariant")
    S = 33 * 45 * 80 + 256
    _, k, v = _torch_inputs(1, 256, S, 24, 5, gpu)
    q = torch.zeros((1, 256, 24, 128), dtype=torch.bfloat16, device=gpu)
    n_valid = S - 137
    out = flash_attention(q, k, v, kv_len=torch.tensor([n_valid], dtype=torch.int32, device=gpu))
    mean = v[:, :n_valid].double().mean(dim=1, keepdim=True)  # (1, 1, H, D)
    err = (out.double() - mean).abs()
    print(f"  max_abs={err.max().item():.3e}", flush=True)
    # all weights are exactly 1 in bf16; only fp32 accumulation and the bf16
    # rounding of a ~3e-3-sized output remain
    assert err.max().item() <= 1e-4


# ---------------------------------------------------- head/query-dependent bias
BIAS_CASES = [
    # B, Sq, Sk, H, seed, bias shape kind
    (2, 200, 200, 4, 60, "t5"),          # (1, H, L, L) relative-position-style bias, scale 1
    (1, 130, 130, 2, 61, "causal"),      # boolean (L, L) lower-triangular mask
    (2, 70, 300, 3, 62, "head_keys"),    # (1, H, 1, Sk): per-head key bias (query-broadcast)
    (2, 96, 515, 2, 63, "t5_padded"),    # (B, H, Sq, Sk) bias + key padding mask
]


@pytest.mark.parametrize("B,Sq,Sk,H,seed,kind", BIAS_CASES)
def test_flash_full_bias_and_masks(gpu, B, Sq, Sk, H, seed, kind):
    """dot_product_attention with a bias or mask that depends on head and/or
    query -- the reference's jax.nn fallback (attention.py:519-533; T5's
    relative bias, t5.py:40-68; causal text attention, cosmos3
    dit_layers.py:114-116) -- against the oracle."""
    from vidax_amd import dot_product_attention
    _say(f"flash bias kind={kind} B={B} Sq={Sq} Sk={Sk} H={H} seed={seed}")
    q, k, v, _ = O.make_flash_inputs(B, Sq, Sk, H, 128, seed)
    rng = np.random.default_rng(seed + 1)
    tq, tk, tv = _t(q, gpu), _t(k, gpu), _t(v, gpu)
    if kind == "t5":
        bias = (2.0 * rng.standard_normal((1, H, Sq, Sk))).astype(np.float32)
        out = dot_product_attention(tq, tk, tv, bias=torch.from_numpy(bias).to(gpu), scale=1.0)
        ref = O.attention(q, k, v, scale=1.0, bias=bias)
    elif kind == "causal":
        causal = np.tril(np.ones((Sq, Sk), bool))
        out = dot_product_attention(tq, tk, tv, mask=torch.from_numpy(causal).to(gpu))
        ref = O.attention(q, k, v, bias=np.where(causal, 0.0, -np.inf))
    elif kind == "head_keys":
        bias = rng.standard_normal((1, H, 1, Sk)).astype(np.float32)
        bias[:, 1, :, 40:90] = -np.inf
        out = dot_product_attention(tq, tk, tv, bias=torch.from_numpy(bias).to(gpu))
        ref = O.attention(q, k, v, bias=bias)
    else:
        bias = rng.standard_normal((B, H, Sq, Sk)).astype(np.float32)
        valid = np.ones((B, 1, 1, Sk), bool)
        valid[0, ..., 400:] = False
        valid[1, ..., 200:260] = False
        out = dot_product_attention(tq, tk, tv, bias=torch.from_numpy(bias).to(gpu),
                                    mask=torch.from_numpy(valid).to(gpu))
        ref = O.attention(q, k, v, bias=bias + np.where(valid, 0.0, -np.inf))
    torch.cuda.synchronize()
    _check(out, ref, kind)


# ------------------------------------------------------------ head dim 64
D64_CASES = [
    # B, Sq, Sk, H, seed, mask
    (1, 128, 128, 2, 70, None),
    (2, 200, 300, 3, 71, None),
    (2, 130, 512, 4, 72, ("kv_len", 20, 512)),
    (2, 96, 515, 2, 73, ("tail_pad", 0, 200)),
]


@pytest.mark.parametrize("B,Sq,Sk,H,seed,mask", D64_CASES)
def test_flash_head_dim_64(gpu, B, Sq, Sk, H, seed, mask):
    from vidax_amd import flash_attention
    _say(f"flash D=64 B={B} Sq={Sq} Sk={Sk} H={H} seed={seed} mask={mask}")
    q, k, v, extra = O.make_flash_inputs(B, Sq, Sk, H, 64, seed, mask)
    kw = {key: torch.from_numpy(val).to(gpu) for key, val in extra.items()}
    out = flash_attention(_t(q, gpu), _t(k, gpu), _t(v, gpu), **kw)
    torch.cuda.synchronize()
    _check(out, O.attention(q, k, v, kv_len=extra.get("kv_len"), key_valid=extra.get("key_valid")), "D=64")


def test_flash_t5_relative_bias_head_dim_64(gpu):
    """UMT5 encoder attention (src/vidax/models/wan/common/t5.py:40-68): head
    dim 64, no softmax scaling, a learned (1, H, L, L) relative-position bias
    plus a (B, 1, 1, L) padding mask, through dot_product_attention."""
    from vidax_amd import dot_product_attention
    _say("flash T5 D=64 L=512 H=8 with relative bias and padding")
    B, L, H = 2, 512, 8
    q, k, v, _ = O.make_flash_inputs(B, L, L, H, 64, 74)
    q, k = q * 0.125, k  # T5 logits are O(1) after its learned projections
    rng = np.random.default_rng(75)
    pos_bias = rng.standard_normal((1, H, L, L)).astype(np.float32)
    pad = np.zeros((B, 1, 1, L), np.float32)
    pad[1, ..., 300:] = -np.inf
    bias = pos_bias + pad
    out = dot_product_attention(_t(q, gpu), _t(k, gpu), _t(v, gpu), bias=torch.from_numpy(bias).to(gpu),
                                scale=1.0)
    torch.cuda.synchronize()
    _check(out, O.attention(O.bf16_round(q), k, v, scale=1.0, bias=bias), "t5")


# ------------------------------------------- 256-query workgroups (8 waves)
# The 8-wave kernel runs for long key sequences on large grids. B=1, H=24,
# Sq=8192 (768 tiles of 256 queries) and Sk=1100 (17 key tiles and a 12-key
# tail) select it while keeping the oracle cheap; sampled query rows (all
# heads) are compared, including the first and last rows.
EIGHT_WAVE_KINDS = ["plain", "kv_len", "key_valid", "key_bias", "all_key_masks", "full_bias"]


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("kind", EIGHT_WAVE_KINDS)
def test_flash_eight_wave_variants(gpu, D, kind):
    from vidax_amd import _lib, dot_product_attention, flash_attention
    B, Sq, Sk, H = 1, 8192, 1100, 24
    mask_kind = {"plain": 0, "kv_len": 0, "key_valid": 1, "key_bias": 2, "all_key_masks": 3, "full_bias": 5}[kind]
    # (a per-(query, key) bias, and key validity with a key bias, always run
    # 128-query workgroups)
    name = f"flash_fwd_kernel<{mask_kind}, {D}, {4 if kind in ('full_bias', 'all_key_masks') else 8}>"
    _say(f"flash 8 waves {name} kind={kind} B={B} Sq={Sq} Sk={Sk} H={H} D={D}")
    seed = 90 + EIGHT_WAVE_KINDS.index(kind) + (0 if D == 128 else 10)
    q, k, v, _ = O.make_flash_inputs(B, Sq, Sk, H, D, seed)
    rng = np.random.default_rng(seed + 1)
    rows = _rows(Sq, 192, seed)
    tq, tk, tv = _t(q, gpu), _t(k, gpu), _t(v, gpu)
    kv_len = np.array([1037], dtype=np.int32)            # ends inside tile 16
    valid = rng.random((B, Sk)) > 0.2
    valid[:, 64:128] = False                             # one whole tile masked
    key_bias = rng.standard_normal((B, Sk)).astype(np.float32)
    key_bias[rng.random((B, Sk)) < 0.05] = -np.inf
    dev = lambda a: torch.from_numpy(a).to(gpu)
    if kind == "plain":
        out = flash_attention(tq, tk, tv)
        ref = O.attention(q[:, rows], k, v)
    elif kind == "kv_len":
        out = flash_attention(tq, tk, tv, kv_len=dev(kv_len))
        ref = O.attention(q[:, rows], k, v, kv_len=kv_len)
    elif kind == "key_valid":
        out = flash_attention(tq, tk, tv, key_valid=dev(valid))
        ref = O.attention(q[:, rows], k, v, key_valid=valid)
    elif kind == "key_bias":
        out = flash_attention(tq, tk, tv, key_bias=dev(key_bias))
        ref = O.attention(q[:, rows], k, v, key_bias=key_bias)
    elif kind == "all_key_masks":
        out = flash_attention(tq, tk, tv, kv_len=dev(kv_len), key_valid=dev(valid), key_bias=dev(key_bias))
        ref = O.attention(q[:, rows], k, v, kv_len=kv_len, key_valid=valid, key_bias=key_bias)
    else:
        # a (B, 1, Sq, Sk) bias shared by all heads plus a boolean key mask
        bias = (0.5 * rng.standard_normal((B, 1, Sq, Sk))).astype(np.float32)
        out = dot_product_attention(tq, tk, tv, bias=dev(bias), mask=dev(valid[:, None, None, :]))
        ref = O.attention(q[:, rows], k, v, key_valid=valid, bias=bias[:, :, rows])
    assert _lib.last_launch() == name, _lib.last_launch()  # the kernel that actually ran
    torch.cuda.synchronize()
    _check(out[:, torch.from_numpy(rows).to(gpu)], ref, f"8 waves {kind} D={D}")


@pytest.mark.parametrize("D", [128, 64])
def test_flash_eight_wave_two_batch_items(gpu, D):
    """8-wave kernel with B=2: per-item kv_len (one inside a tile, one
    below Sk by a whole tile and more) and key_valid holes, sampled rows of
    both items."""
    from vidax_amd import _lib, flash_attention
    B, Sq, Sk, H = 2, 4096, 1100, 24
    name = f"flash_fwd_kernel<1, {D}, 8>"
    _say(f"flash 8 waves B=2 {name} Sq={Sq} Sk={Sk} H={H} D={D}")
    seed = 120 + (0 if D == 128 else 1)
    q, k, v, _ = O.make_flash_inputs(B, Sq, Sk, H, D, seed)
    rng = np.random.default_rng(seed + 1)
    kv_len = np.array([1037, 655], dtype=np.int32)
    valid = rng.random((B, Sk)) > 0.25
    valid[1, 128:192] = False
    rows = _rows(Sq, 160, seed)
    dev = lambda a: torch.from_numpy(a).to(gpu)
    out = flash_attention(_t(q, gpu), _t(k, gpu), _t(v, gpu), kv_len=dev(kv_len), key_valid=dev(valid))
    assert _lib.last_launch() == name, _lib.last_launch()
    torch.cuda.synchronize()
    ref = O.attention(q[:, rows], k, v, kv_len=kv_len, key_valid=valid)
    _check(out[:, torch.from_numpy(rows).to(gpu)], ref, f"8 waves B=2 D={D}")


@pytest.mark.parametrize("shape", [(2, 300, 700, 3), (1, 8192, 1100, 24)], ids=["pairs", "8 waves"])
@pytest.mark.parametrize("D", [128, 64])
def test_flash_dominant_key_bias(gpu, shape, D):
    """A key bias that dominates the logits (+-40, runs of -inf in the middle
    of the sequence as in Cosmos3's text padding) with a small scale (0.02):
    the bias enters the QK^T accumulator as bias / scale (up to 2000), and
    the reference point has to follow the bias, not q.k."""
    from vidax_amd import _lib, flash_attention
    B, Sq, Sk, H = shape
    # (18 query tiles of 11 key tiles run as pairs)
    name = f"flash_pair_kernel<2, {D}>" if Sq < 1000 else f"flash_fwd_kernel<2, {D}, 8>"
    _say(f"flash dominant key bias {name} B={B} Sq={Sq} Sk={Sk} H={H} D={D}")
    seed = 130 + (0 if D == 128 else 1) + (0 if Sq < 1000 else 2)
    q, k, v, _ = O.make_flash_inputs(B, Sq, Sk, H, D, seed)
    rng = np.random.default_rng(seed + 1)
    bias = (40.0 * rng.uniform(-1.0, 1.0, (B, Sk))).astype(np.float32)
    bias[:, Sk // 3:Sk // 3 + 150] = -np.inf          # a padded run mid-sequence
    bias[rng.random((B, Sk)) < 0.05] = -np.inf
    rows = _rows(Sq, min(Sq, 160), seed)
    out = flash_attention(_t(q, gpu), _t(k, gpu), _t(v, gpu), scale=0.02,
                          key_bias=torch.from_numpy(bias).to(gpu))
    assert _lib.last_launch() == name, _lib.last_launch()
    torch.cuda.synchronize()
    ref = O.attention(q[:, rows], k, v, scale=0.02, key_bias=bias)
    _check(out[:, torch.from_numpy(rows).to(gpu)], ref, f"dominant key bias {name}")


# ----------------------------------------- key-axis broadcast of bias / mask
def test_flash_bias_and_mask_broadcast_along_keys(gpu):
    """A (1, H, Sq, 1) bias and a (B, 1, Sq, 1) boolean mask broadcast over the
    keys as jnp.broadcast_to does (src/vidax/core/attention.py:282,533): a
    per-(head, query) constant bias leaves the softmax unchanged, and a
    per-(batch, query) False masks every key of that query row."""
    from vidax_amd import dot_product_attention
    _say("flash bias (1,H,Sq,1) and mask (B,1,Sq,1)")
    B, Sq, Sk, H = 2, 90, 300, 3
    q, k, v, _ = O.make_flash_inputs(B, Sq, Sk, H, 128, 140)
    rng = np.random.default_rng(141)
    tq, tk, tv = _t(q, gpu), _t(k, gpu), _t(v, gpu)
    bias = (3.0 * rng.standard_normal((1, H, Sq, 1))).astype(np.float32)
    out = dot_product_attention(tq, tk, tv, bias=torch.from_numpy(bias).to(gpu))
    torch.cuda.synchronize()
    _check(out, O.attention(q, k, v, bias=bias), "bias (1,H,Sq,1)")
    _check(out, O.attention(q, k, v), "bias (1,H,Sq,1) = no bias")
    mask = np.ones((B, 1, Sq, 1), bool)
    mask[0, 0, 10:20, 0] = False
    mask[1, 0, 50, 0] = False
    out = dot_product_attention(tq, tk, tv, mask=torch.from_numpy(mask).to(gpu))
    torch.cuda.synchronize()
    o = out.float().cpu().numpy()
    keep = np.broadcast_to(mask[:, 0, :, 0][:, :, None, None], o.shape)
    # rows with every key masked are written as zeros (the library's documented
    # choice where the reference's softmax would give 0/0)
    assert (o[~keep] == 0).all()
    ref = O.attention(q, k, v)
    err = np.abs(o - ref)[keep]
    assert err.max() <= MAX_ABS and err.mean() <= MEAN_ABS


# ------------------------------------------- forced tile sizes (env override)
_FORCED = """
import sys, json
sys.path.insert(0, {root!r})
import numpy as np, torch
from oracle import attention_oracle as O
from vidax_amd import _lib, flash_attention
B, Sq, Sk, H, D, seed = {shape}
q, k, v, _ = O.make_flash_inputs(B, Sq, Sk, H, D, seed)
rows = np.unique(np.linspace(0, Sq - 1, 96).astype(int))
t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda().to(torch.bfloat16)
kv_len = np.array([Sk - 37] * B, np.int32)
out = flash_attention(t(q), t(k), t(v), kv_len=torch.from_numpy(kv_len).cuda())
name = _lib.last_launch()
torch.cuda.synchronize()
ref = O.attention(q[:, rows], k, v, kv_len=kv_len)
err = np.abs(out[:, torch.from_numpy(rows).cuda()].float().cpu().numpy() - ref)
print(json.dumps(dict(name=name, max=float(err.max()), mean=float(err.mean()))))
"""


@pytest.mark.parametrize("block_q,shape", [
    (256, (1, 700, 1500, 4, 128, 150)),    # the table picks 128-query workgroups here
    (128, (1, 8192, 1100, 24, 128, 151)),  # and 256-query ones here
    (256, (2, 300, 520, 3, 64, 152)),
])
def test_flash_forced_block_sizes(gpu, block_q, shape):
    """VIDAX_FLASH_BLOCK_SIZES forces the query tile (read once per process,
    so each case runs in a fresh interpreter); the forced kernel launches and
    matches the oracle."""
    import json
    import os
    import subprocess
    import sys
    _say(f"flash forced VIDAX_FLASH_BLOCK_SIZES={block_q},64,64 shape={shape}")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, VIDAX_FLASH_BLOCK_SIZES=f"{block_q},64,64")
    res = subprocess.run([sys.executable, "-c", _FORCED.format(root=root, shape=shape)], env=env,
                         stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=240)
    assert res.returncode == 0, res.stdout[-2000:]
    r = json.loads(res.stdout.strip().splitlines()[-1])
    print(f"  {r}", flush=True)
    # (small grids also split their keys: the split form of the same kernel)
    assert r["name"] in (f"flash_fwd_kernel<0, {shape[4]}, {block_q // 32}>",
                         f"flash_fwd_split_kernel<0, {shape[4]}, {block_q // 32}>"), r["name"]
    assert r["max"] <= MAX_ABS and r["mean"] <= MEAN_ABS


# ------------------------------------------- persistent short-key kernel
STREAM_CASES = [
    # B, Sq, Sk, H, D, kv_len, seed
    (2, 32768, 512, 16, 128, [432, 148], 160),   # seven- and three-tile items (the cross-attention mix)
    (3, 15000, 300, 24, 128, [0, 65, 300], 161), # an empty batch item, two-tile items, ragged queries
    (2, 20000, 130, 26, 128, [1, 64], 162),      # one-tile items
    (1, 65536, 1024, 16, 128, None, 163),        # sixteen tiles, no kv_len
    (2, 32760, 512, 16, 64, [512, 20], 164),     # head dim 64
    (2, 16384, 256, 32, 128, [0, 0], 166),       # no keys at all: zero rows only
    (8, 8192, 1024, 16, 128, [0, 1, 64, 1000, 0, 37, 1024, 700], 167),  # eight mixed batch items
]


@pytest.mark.parametrize("B,Sq,Sk,H,D,kv,seed", STREAM_CASES)
def test_flash_stream_kernel(gpu, B, Sq, Sk, H, D, kv, seed):
    """The persistent short-key kernel (one workgroup per CU running the key
    tiles of its items as one stream): rows at every position of a 256-query
    tile, and the first and last rows, against the oracle (zero rows for
    kv_len 0); and bit for bit the output of the 128-query kernel given the
    same keys as a boolean key mask."""
    from vidax_amd import _lib, dot_product_attention, flash_attention
    _say(f"flash stream B={B} Sq={Sq} Sk={Sk} H={H} D={D} kv_len={kv} seed={seed}")
    g = torch.Generator(device=gpu)
    g.manual_seed(seed)
    q, k, v = (torch.randn((B, n, H, D), generator=g, device=gpu, dtype=torch.float32).to(torch.bfloat16)
               for n in (Sq, Sk, Sk))
    kv_t = None if kv is None else torch.tensor(kv, dtype=torch.int32, device=gpu)
    out = flash_attention(q, k, v, kv_len=kv_t)
    torch.cuda.synchronize()
    assert _lib.last_launch() == f"flash_stream_kernel<{D}>", _lib.last_launch()
    rows = _residue_rows(Sq, 1, seed)
    kv_np = None if kv is None else np.array(kv, np.int32)
    ref = O.attention_rows(_np(q), _np(k), _np(v), rows, kv_len=kv_np)
    _check(out[:, torch.from_numpy(rows).to(gpu)], ref, "stream rows")
    if kv is not None:
        valid = torch.arange(Sk, device=gpu)[None, :] < kv_t[:, None]
        out2 = dot_product_attention(q, k, v, mask=valid[:, None, None, :])
        torch.cuda.synchronize()
        assert _lib.last_launch() == f"flash_fwd_kernel<1, {D}, 4>", _lib.last_launch()
        assert torch.equal(out, out2)


def test_flash_stream_kernel_strided_views(gpu):
    """q, k and v as views into wider rows (the persistent kernel's copies
    use each tensor's own strides)."""
    from vidax_amd import _lib, flash_attention
    _say("flash stream strided views B=2 Sq=20000 Sk=200 H=26")
    B, Sq, Sk, H, D = 2, 20000, 200, 26, 128
    g = torch.Generator(device=gpu)
    g.manual_seed(165)
    qw = torch.randn((B, Sq, H, 2 * D), generator=g, device=gpu, dtype=torch.float32).to(torch.bfloat16)
    kvw = torch.randn((B, Sk, 3, H, D), generator=g, device=gpu, dtype=torch.float32).to(torch.bfloat16)
    q, k, v = qw[..., D:], kvw[:, :, 0], kvw[:, :, 2]
    kv = np.array([200, 77], np.int32)
    out = flash_attention(q, k, v, kv_len=torch.from_numpy(kv).to(gpu))
    torch.cuda.synchronize()
    assert _lib.last_launch() == "flash_stream_kernel<128>", _lib.last_launch()
    rows = _residue_rows(Sq, 1, 165)
    ref = O.attention_rows(_np(q), _np(k), _np(v), rows, kv_len=kv)
    _check(out[:, torch.from_numpy(rows).to(gpu)], ref, "stream strided rows")
    out_c = flash_attention(q.contiguous(), k.contiguous(), v.contiguous(), kv_len=torch.from_numpy(kv).to(gpu))
    assert torch.equal(out, out_c)


def test_flash_stream_kernel_last_row_after_late_rescale(gpu):
    """Ragged Sq: the last 256-query tile holds queries past Sq, whose lanes
    repeat row Sq-1's query. Only the wave that owns row Sq-1 may store it.
    Built so that the owner's wave takes the rare rescale in the last key
    tile (another of its queries, row Sq-2, scores one late key far above
    everything), and row Sq-1 itself has a new, moderate maximum in that
    tile: the owner raises row Sq-1's reference point there, the waves that
    only hold copies of row Sq-1 do not, so their bf16 probabilities (and
    stores) would differ. Every row must equal, bit for bit, the 128-query
    kernel's (same waves: each row stored once, by its owner)."""
    from vidax_amd import _lib, dot_product_attention, flash_attention
    B, Sq, Sk, H, D, kv, seed = 1, 65436, 512, 16, 128, 500, 168
    _say(f"flash stream ragged Sq={Sq} late rescale in the owner's wave, H={H} kv_len={kv}")
    g = torch.Generator(device=gpu)
    g.manual_seed(seed)
    q, k, v = (torch.randn((B, n, H, D), generator=g, device=gpu, dtype=torch.float32) for n in (Sq, Sk, Sk))
    js = 470                                          # a key in the last tile (keys 448..499)
    ks = k[0, js]                                     # (H, D)
    nrm2 = (ks * ks).sum(-1, keepdim=True)
    scale = D ** -0.5
    # row Sq-2: logit 20 on key js (2^24 above its reference point: the rare path)
    q[0, Sq - 2] = ks * (20.0 / (scale * nrm2))
    # row Sq-1: logit 4.5 on key js, all its other logits ~N(0, 0.4^2): a new
    # maximum in the last tile, probability sum well below 2^8 (no rescale of its own)
    q[0, Sq - 1] = ks * (4.5 / (scale * nrm2))
    q, k, v = (x.to(torch.bfloat16) for x in (q, k, v))
    kv_t = torch.tensor([kv], dtype=torch.int32, device=gpu)
    out = flash_attention(q, k, v, kv_len=kv_t)
    torch.cuda.synchronize()
    assert _lib.last_launch() == "flash_stream_kernel<128>", _lib.last_launch()
    valid = torch.arange(Sk, device=gpu)[None, :] < kv_t[:, None]
    out2 = dot_product_attention(q, k, v, mask=valid[:, None, None, :])
    torch.cuda.synchronize()
    assert _lib.last_launch() == "flash_fwd_kernel<1, 128, 4>", _lib.last_launch()
    tail = slice(Sq - 64, Sq)
    print(f"  last rows equal: {torch.equal(out[:, tail], out2[:, tail])}", flush=True)
    assert torch.equal(out, out2)
    rows = np.array([0, Sq - 300, Sq - 3, Sq - 2, Sq - 1])
    ref = O.attention_rows(_np(q), _np(k), _np(v), rows, kv_len=np.array([kv], np.int32))
    _check(out[:, torch.from_numpy(rows).to(gpu)], ref, "stream ragged rows")


# ------------------------------------------------ key split of the last round
def _plain_flash(q, k, v, kw, scale=None):
    """The same call through vx_flash_attn_fwd, which never splits."""
    import ctypes
    from vidax_amd import _lib
    B, Sq, H, D = q.shape
    Sk = k.shape[1]
    out = torch.empty_like(q)
    kvl = kw.get("kv_len")
    # rows of whole 64-key tiles, padded with invalid / -inf keys
    pad = lambda x, dtype, fill: torch.nn.functional.pad(x.to(dtype), (0, -Sk % 64), value=fill).contiguous()
    kvd = pad(kw["key_valid"].to(torch.bool), torch.uint8, 0) if "key_valid" in kw else None
    kbs = pad(kw["key_bias"], torch.float32, float("-inf")) if "key_bias" in kw else None
    stride = (kvd if kvd is not None else kbs).shape[1] if (kvd is not None or kbs is not None) else 0
    rc = _lib.lib().vx_flash_attn_fwd(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
        kvl.data_ptr() if kvl is not None else None, kvd.data_ptr() if kvd is not None else None,
        kbs.data_ptr() if kbs is not None else None, stride, B, Sq, Sk, H, D, None, None, None, None,
        ctypes.c_float(scale if scale is not None else D ** -0.5),
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    _lib.raise_for(rc)
    return out


SPLIT_CASES = [
    # B, Sq, Sk, H, D, seed, mask, expected kernel
    (1, 2048, 1500, 3, 128, 160, None, "flash_pair_split_kernel<0, 128>"),            # every item split, as pairs
    (2, 700, 2100, 2, 128, 161, ("kv_len", 0, 2100), "flash_pair_split_kernel<0, 128>"),
    (1, 900, 1600, 3, 64, 162, ("tail_pad", 0, 200), "flash_pair_split_kernel<1, 64>"),
    (1, 900, 1100, 3, 64, 162, ("tail_pad", 0, 200), "flash_pair_kernel<1, 64>"),     # 18 key tiles: one pair
    # 4 waves, above one workgroup per CU: 516 items (4 split), 600 items (88 split)
    (1, 5400, 1100, 12, 128, 164, None, "flash_fwd_split_kernel<0, 128, 4>"),
    (2, 3200, 1100, 12, 64, 165, ("tail_pad", 0, 200), "flash_fwd_split_kernel<1, 64, 4>"),
    (2, 3200, 1100, 12, 128, 166, ("kv_len", 0, 1100), "flash_fwd_split_kernel<0, 128, 4>"),
    (1, 8192, 2048, 25, 128, 163, None, "flash_fwd_split_kernel<0, 128, 8>"),         # 800 items: 32 split
]


@pytest.mark.parametrize("B,Sq,Sk,H,D,seed,mask,name", SPLIT_CASES)
def test_flash_key_split(gpu, B, Sq, Sk, H, D, seed, mask, name):
    """Query tiles of the grid's last round split over the two key halves
    (fp32 partials merged by a second kernel) against the oracle, and
    against the unsplit kernel on the same inputs."""
    from vidax_amd import _lib, flash_attention
    _say(f"flash key split B={B} Sq={Sq} Sk={Sk} H={H} D={D} mask={mask}")
    q, k, v, extra = O.make_flash_inputs(B, Sq, Sk, H, D, seed, mask)
    kw = {key: torch.from_numpy(val).to(gpu) for key, val in extra.items()}
    if mask is not None and mask[0] == "kv_len":
        kw["kv_len"][0] = 700          # item 0 has no key in the second half (keys >= 1024)
        extra["kv_len"][0] = 700
    tq, tk, tv = _t(q, gpu), _t(k, gpu), _t(v, gpu)
    out = flash_attention(tq, tk, tv, **kw)
    assert _lib.last_launch() == name, _lib.last_launch()
    plain = _plain_flash(tq, tk, tv, kw)
    torch.cuda.synchronize()
    rows = _rows(Sq, min(Sq, 256), seed) if Sq > 2048 else np.arange(Sq)
    ref = O.attention(q[:, rows], k, v, kv_len=extra.get("kv_len"), key_valid=extra.get("key_valid"))
    _check(out[:, torch.from_numpy(rows).to(gpu)], ref, "split vs oracle")
    d = (out.float() - plain.float()).abs()
    print(f"  split vs unsplit: max {d.max().item():.3e} mean {d.mean().item():.3e}", flush=True)
    assert d.max().item() <= MAX_ABS and d.mean().item() <= MEAN_ABS


def test_flash_key_bias_is_not_split(gpu):
    """A shape whose grid would split its keys runs unsplit when a key bias is
    given (-inf runs in both halves of the keys), and matches the oracle."""
    from vidax_amd import _lib, flash_attention
    _say("flash key split + key_bias")
    B, Sq, Sk, H, D = 1, 1024, 1800, 4, 128
    q, k, v, _ = O.make_flash_inputs(B, Sq, Sk, H, D, 170)
    rng = np.random.default_rng(171)
    bias = (4.0 * rng.standard_normal((B, Sk))).astype(np.float32)
    bias[:, 100:300] = -np.inf
    bias[:, 1200:1250] = -np.inf
    tq, tk, tv = _t(q, gpu), _t(k, gpu), _t(v, gpu)
    kb = torch.from_numpy(bias).to(gpu)
    out = flash_attention(tq, tk, tv, key_bias=kb)
    assert _lib.last_launch() == "flash_pair_kernel<2, 128>", _lib.last_launch()
    plain = _plain_flash(tq, tk, tv, {"key_bias": kb})
    torch.cuda.synchronize()
    _check(out, O.attention(q, k, v, key_bias=bias), "split key_bias vs oracle")
    d = (out.float() - plain.float()).abs()
    print(f"  split vs unsplit: max {d.max().item():.3e} mean {d.mean().item():.3e}", flush=True)
    assert d.max().item() <= MAX_ABS and d.mean().item() <= MEAN_ABS


@pytest.mark.parametrize("pattern", ["prefix", "holes", "none_valid"])
def test_masked_self_attention_key_valid_patterns(gpu, pattern):
    """masked_self_attention hands key_valid to the validity kernel with
    kv_len = last valid key + 1 and never inspects the mask on the host; the
    kernel classifies each 64-key tile (all valid: unmasked path). A prefix
    mask must give the same result as kv_len alone (the unmasked kernel), and
    every pattern agrees with the oracle."""
    from vidax_amd import _lib, flash_attention, masked_self_attention
    _say(f"masked_self_attention key_valid pattern={pattern}")
    B, S, H, D = 2, 700, 4, 128
    q, k, v = _torch_inputs(B, S, S, H, 41, gpu)
    valid = torch.ones((B, S), dtype=torch.bool, device=gpu)
    if pattern == "prefix":
        valid[0, 513:] = False
        valid[1, 90:] = False
    elif pattern == "holes":
        valid[0, 100:130] = False
        valid[1, 650:] = False
    else:
        valid[1, :] = False
    out = masked_self_attention(q, k, v, key_valid=valid).reshape(B, S, H, D)
    launched = _lib.last_launch()
    assert launched == "flash_pair_kernel<1, 128>", launched
    rows = _rows(S, 64, 41)
    ref = O.attention_rows(_np(q), _np(k), _np(v), rows, key_valid=_np(valid).astype(bool))
    _check(out[:, torch.from_numpy(rows).to(gpu)], ref, f"key_valid {pattern} ({launched})")
    if pattern != "holes":
        last = (valid * torch.arange(1, S + 1, device=gpu)).amax(dim=1)
        by_len = flash_attention(q, k, v, kv_len=last)
        torch.cuda.synchronize()
        assert _lib.last_launch() == "flash_pair_kernel<0, 128>", _lib.last_launch()
        same = torch.equal(out, by_len)
        d = (out.float() - by_len.float()).abs()
        print(f"  validity kernel vs kv_len alone: equal={same} max {d.max().item():.3e}", flush=True)
        assert d.max().item() <= 1e-2 and d.mean().item() <= 1e-4, (d.max().item(), d.mean().item())


@pytest.mark.parametrize("form", ["pure_hole", "pure_prefix", "general", "zero"])
def test_dot_product_attention_key_bias_forms(gpu, form):
    """A (B,1,1,Sk) key bias stays a key bias (no host inspection): the
    kernel starts the accumulators of all-zero bias tiles at zero and adds
    the bias elsewhere. Cosmos3's padding bias (0 / -inf: a hole, or a valid
    prefix) must equal the same keys given as a validity mask; a general
    bias and an all-zero one agree with the oracle (the zero bias with the
    unmasked kernel)."""
    from vidax_amd import _lib, dot_product_attention
    _say(f"dot_product_attention key bias form={form}")
    B, S, H, D = 2, 640, 4, 128
    q, k, v = _torch_inputs(B, S, S, H, 43, gpu)
    bias = torch.zeros((B, S), dtype=torch.float32, device=gpu)
    if form == "pure_hole":
        bias[:, 200:260] = float("-inf")
    elif form == "pure_prefix":
        bias[0, 500:] = float("-inf")
        bias[1, 37:] = float("-inf")
    elif form == "general":
        bias = torch.randn((B, S), generator=torch.Generator(device=gpu).manual_seed(43), device=gpu)
        bias[:, 300:333] = float("-inf")
    out = dot_product_attention(q, k, v, bias=bias[:, None, None, :])
    launched = _lib.last_launch()
    assert launched == "flash_pair_kernel<2, 128>", launched
    rows = _rows(S, 64, 43)
    ref = O.attention_rows(_np(q), _np(k), _np(v), rows, key_bias=_np(bias))
    _check(out[:, torch.from_numpy(rows).to(gpu)], ref, f"key bias form {form} ({launched})")
    if form != "general":
        as_mask = dot_product_attention(q, k, v, mask=(bias > float("-inf"))[:, None, None, :])
        torch.cuda.synchronize()
        assert _lib.last_launch() == "flash_pair_kernel<1, 128>", _lib.last_launch()
        d = (out.float() - as_mask.float()).abs()
        print(f"  key bias vs validity mask: equal={torch.equal(out, as_mask)} max {d.max().item():.3e}",
              flush=True)
        assert d.max().item() <= 1e-2 and d.mean().item() <= 1e-4, (d.max().item(), d.mean().item())


# ------------------------------------- two groups of waves per query tile (pairs)
PAIR_CASES = [
    # B, Sq, Sk, H, D, mask (grids of at most one workgroup per CU)
    (1, 130, 384, 2, 64, None),                       # 6 tiles: the first pair at head dim 64
    (1, 70, 320, 2, 64, None),                        # 5 tiles: one group
    (2, 129, 449, 3, 64, ("kv_len", 449, 1)),         # an odd tile count; one key: group 1 without tiles
    (2, 33, 640, 2, 128, ("kv_len", 0, 129)),         # no key; three tiles, two and one
    (1, 128, 640, 2, 128, None),                      # 10 tiles: the first pair at head dim 128
    (1, 200, 705, 2, 128, ("tail_pad", 200)),         # 12 tiles, key validity with an empty tail
    (1, 140, 1537, 2, 128, None),                     # 25 tiles: key halves on two pairs
    (2, 140, 1537, 2, 64, ("kv_len", 1000, 700)),     # the second key half empty for one item
]


@pytest.mark.parametrize("B,Sq,Sk,H,D,mask", PAIR_CASES)
@pytest.mark.parametrize("kind", ["plain", "key_bias", "full_bias"])
def test_flash_pairs(gpu, B, Sq, Sk, H, D, mask, kind):
    """Grids that leave CUs idle run two groups of four waves per query tile,
    each over half of the key tiles, merged in LDS: against the oracle at the
    edges of the rule and of the halves, with every mask form that runs pairs."""
    from vidax_amd import _lib, flash_attention
    _say(f"flash pairs B={B} Sq={Sq} Sk={Sk} H={H} D={D} mask={mask} {kind}")
    q, k, v, extra = O.make_flash_inputs(B, Sq, Sk, H, D, 190)
    rng = np.random.default_rng(191)
    if mask is not None and mask[0] == "kv_len":
        extra["kv_len"] = np.array(mask[1:], np.int32)
    elif mask is not None:
        extra["key_valid"] = np.broadcast_to(np.arange(Sk) < Sk - mask[1], (B, Sk)).copy()
    if kind == "key_bias":
        if "key_valid" in extra:
            pytest.skip("validity together with a key bias runs one group")
        extra["key_bias"] = rng.standard_normal((B, Sk)).astype(np.float32)
        extra["key_bias"][:, Sk // 3:Sk // 3 + 70] = -np.inf
        extra["key_bias"][:, 0] = 0.0
    if kind == "full_bias":
        extra["bias"] = rng.standard_normal((1, H, Sq, Sk)).astype(np.float32)
        extra["bias"][..., 1::7] = -np.inf
    out = flash_attention(_t(q, gpu), _t(k, gpu), _t(v, gpu),
                          **{n: torch.from_numpy(x).to(gpu) for n, x in extra.items()})
    launched = _lib.last_launch()
    torch.cuda.synchronize()
    tiles = -(-Sk // 64)
    m = (1 if "key_valid" in extra else 0) | (2 if "key_bias" in extra else 0) | (4 if "bias" in extra else 0)
    if tiles < (6 if D == 64 else 16 if m & 4 else 10):
        want = f"flash_fwd_kernel<{m}, {D}, 4>"
    else:
        want = f"flash_pair_{'split_' if tiles >= (24 if D == 64 else 20) and not m & 6 else ''}kernel<{m}, {D}>"
    assert launched == want, (launched, want)
    if "bias" in extra:
        extra["bias"] = np.broadcast_to(extra["bias"], (B, H, Sq, Sk))
    ref = O.attention(q, k, v, **extra)
    if "kv_len" in extra and (extra["kv_len"] == 0).any():
        assert (out[0] == 0).all()
        out, ref = out[1:], ref[1:]
    _check(out, ref, "oracle")


@pytest.mark.parametrize("D,Sk,short,mask", [
    (128, 640, 5, None),          # 10 key tiles: pairs; items of 5 and fewer
    (128, 1024, 9, None),         # one tile below the rule
    (64, 384, 5, None),
    (128, 704, 3, "key_valid"),
    (64, 448, 4, "key_bias"),
    (64, 512, 5, "full_bias"),
])
def test_flash_pairs_of_short_items(gpu, D, Sk, short, mask):
    """Where kv_len ends an item's keys below the pairs' key tiles, one group
    of waves takes them all: bit for bit the call on `short` key tiles, which
    runs flash_fwd_kernel. A long item of the same call still runs two."""
    from vidax_amd import _lib, flash_attention
    _say(f"flash pairs of short items D={D} Sk={Sk} {short} tiles {mask}")
    B, Sq, H, n = 3, 150, 2, 64 * short
    q, k, v, _ = O.make_flash_inputs(B, Sq, Sk, H, D, 210)
    q, k, v = _t(q, gpu), _t(k, gpu), _t(v, gpu)
    kv = torch.tensor([n - 7, 0 if mask is None else n - 64, Sk], dtype=torch.int32, device=gpu)
    g = torch.Generator(device=gpu).manual_seed(211)
    kw = {}
    if mask == "key_valid":
        kw["key_valid"] = torch.rand((B, Sk), generator=g, device=gpu) < 0.7
    elif mask == "key_bias":
        kw["key_bias"] = torch.randn((B, Sk), generator=g, device=gpu)
    elif mask == "full_bias":
        kw["bias"] = torch.randn((1, H, Sq, Sk), generator=g, device=gpu)
    out = flash_attention(q, k, v, kv_len=kv, **kw)
    assert _lib.last_launch().startswith("flash_pair_kernel<"), _lib.last_launch()
    cut = {name: x[..., :n].contiguous()[:2 if x.shape[0] == B else 1] for name, x in kw.items()}
    ref = flash_attention(q[:2], k[:2, :n].contiguous(), v[:2, :n].contiguous(), kv_len=kv[:2], **cut)
    assert _lib.last_launch().startswith("flash_fwd_kernel<"), _lib.last_launch()
    torch.cuda.synchronize()
    assert torch.equal(out[:2], ref)
    np_kw = {name: x.cpu().numpy() for name, x in kw.items()}
    if "bias" in np_kw:
        np_kw["bias"] = np.broadcast_to(np_kw["bias"], (B, H, Sq, Sk))
    _check(out[2:], O.attention(*(_np(x) for x in (q, k, v)), kv_len=kv.cpu().numpy().clip(min=1), **np_kw)[2:],
           "long item vs oracle")
