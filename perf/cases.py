"""Performance cases of the attention kernels: what a video diffusion
transformer (and its text encoder and VAE) calls, through the public entry
points of vidax_amd, from the smallest calls to the largest.

A case is a dict of plain values; `listed()` holds the named ones, `draw(rng)`
makes another one of the same ranges. Kinds:

masked    masked_self_attention with a key-validity mask whose last keys are
          padding: joint video + text self-attention, the token refiner
text      dot_product_attention of a text encoder: a (1, H, L, L)
          relative-position bias with a (B, 1, 1, L) padding mask, or a causal
          (1, 1, L, L) boolean mask
self      dot_product_attention without a mask: video self-attention
cross     video queries against text keys: flash_attention with kv_len (padded
          prompts), or dot_product_attention over all keys
key_bias  dot_product_attention with a (B, 1, 1, S) additive bias, 0 on valid
          keys and -inf on a run of padding in the middle of the sequence
na        neighborhood_attention_3d, q scaled by the caller
na_block  the neighbourhood block: k through na3d_qk_norm_rope, then
          na3d_block_attention with q prepared inside it
prologue  qk_norm_rope of q and of k: RMSNorm over the projected row, 3D RoPE
"""
import math

import torch

import vidax_amd

BF16 = torch.bfloat16


def listed():
    return [
        # the token refiner over a padded prompt, two prompts (guidance)
        dict(name="refiner_256", kind="masked", B=2, S=256, H=24, D=128, pad0=0, pad1=177),
        # a T5-style encoder layer over two padded prompts
        dict(name="text_512", kind="text", B=2, S=512, H=8, D=64, causal=False, pad0=0, pad1=200),
        # one latent frame of 30 x 52 tokens, 12 heads
        dict(name="self_1560", kind="self", B=1, S=1560, H=12, D=128),
        # five such frames
        dict(name="self_7800", kind="self", B=1, S=7800, H=12, D=128),
        # 21 frames, 40 heads: the headline self-attention
        dict(name="self_32760", kind="self", B=1, S=32760, H=40, D=128),
        # the same video tokens against two padded prompts
        dict(name="cross_32760x512", kind="cross", B=2, S=32760, Sk=512, H=40, D=128, kv0=432, kv1=148),
        # joint attention over 33 x 45 x 80 video and 256 text tokens
        dict(name="joint_119056", kind="masked", B=1, S=119056, H=24, D=128, pad0=137, pad1=0),
        # packed sequence with its text padding in the middle
        dict(name="key_bias_8192", kind="key_bias", B=1, S=8192, H=24, D=128, hole=200),
        # neighbourhood attention on 21 x 45 x 80 tokens
        dict(name="na_21x45x80", kind="na", B=1, T=21, Y=45, X=80, H=24, D=128, kt=3, ky=7, kx=7),
        # a block of the VAE's last stage and one of its first
        dict(name="na_block_33x88x160", kind="na_block", B=1, T=33, Y=88, X=160, H=4, D=64, kt=11, ky=11, kx=11),
        dict(name="na_block_5x22x40", kind="na_block", B=1, T=5, Y=22, X=40, H=16, D=64, kt=3, ky=7, kx=7),
        # q and k of the headline self-attention
        dict(name="prologue_32760", kind="prologue", B=1, T=21, Y=30, X=52, H=40, D=128),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["masked", "text", "self", "self", "cross", "key_bias", "na", "na", "na_block", "prologue"])
    B = rng.choice([1, 1, 2])
    if kind in ("masked", "self", "key_bias"):
        while True:
            c = dict(kind=kind, B=B, S=_log_int(rng, 100, 60000), H=rng.choice([8, 12, 16, 24, 30, 40]),
                     D=rng.choice([128, 128, 64]))
            if c["B"] * c["S"] * c["S"] * c["H"] < 32760 * 32760 * 40:
                break
        if kind == "masked":
            c.update(pad0=rng.randint(0, min(200, c["S"] - 20)), pad1=rng.randint(0, min(200, c["S"] - 20)))
        if kind == "key_bias":
            c.update(hole=rng.randint(1, min(300, c["S"] // 2)))
        return c
    if kind == "text":
        S = _log_int(rng, 32, 512)
        return dict(kind=kind, B=B, S=S, H=rng.choice([8, 12, 16, 32, 64]), D=rng.choice([64, 64, 128]),
                    causal=rng.random() < 0.3, pad0=rng.randint(0, S // 2), pad1=rng.randint(0, S // 2))
    if kind == "cross":
        Sk = rng.choice([77, 226, 256, 257, 512, rng.randint(20, 1024)])
        padded = rng.random() < 0.5
        return dict(kind=kind, B=B, S=_log_int(rng, 500, 80000), Sk=Sk, H=rng.choice([8, 12, 16, 24, 40]), D=128,
                    kv0=rng.randint(20, Sk) if padded else 0, kv1=rng.randint(20, Sk) if padded else 0)
    if kind == "prologue":
        return dict(kind=kind, B=B, T=rng.randint(1, 33), Y=rng.randint(8, 48), X=rng.randint(14, 80),
                    H=rng.choice([12, 16, 24, 40]), D=128)
    while True:
        kt, ky, kx = rng.choice([(3, 5, 5), (3, 7, 7), (3, 7, 7), (11, 11, 11), (11, 11, 11), (5, 9, 9), (1, 7, 7),
                                 (3, 11, 15), (3, 7, 31)])
        c = dict(kind=kind, B=1, T=rng.randint(2, 33), Y=_log_int(rng, 8, 90), X=_log_int(rng, 14, 160),
                 H=rng.choice([4, 8, 12, 16, 24]), D=rng.choice([64, 64, 128]), kt=kt, ky=ky, kx=kx)
        n = c["T"] * c["Y"] * c["X"] * c["H"] * c["D"]
        if n <= 21 * 45 * 80 * 24 * 128 and n * min(kt, c["T"]) * min(ky, c["Y"]) * kx <= 33 * 88 * 160 * 4 * 64 * 1331:
            return c


# ------------------------------------------------------------------ the inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, std=1.0):
    x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    return (x * std if std != 1.0 else x).to(BF16)


def _valid(case):
    """(B, S) bool, the last pad keys of each batch item invalid."""
    S = case["S"]
    lens = [S - case["pad0"], S - case["pad1"]][:case["B"]]
    return torch.arange(S, device="cuda")[None, :] < torch.tensor(lens, device="cuda")[:, None]


def prepare(case, seed):
    g = _gen(seed)
    kind, B, H, D = case["kind"], case["B"], case["H"], case["D"]
    st = dict(case=case)
    if kind in ("na", "na_block"):
        shape = (B, case["T"], case["Y"], case["X"], H, D)
        st["window"] = (case["kt"], case["ky"], case["kx"])
        if kind == "na":
            st["q"], st["k"], st["v"] = _randn(g, *shape, std=D ** -0.5), _randn(g, *shape), _randn(g, *shape)
        else:
            st["q"], st["k"], st["v"] = _randn(g, *shape, std=2.0), _randn(g, *shape, std=2.0), _randn(g, *shape)
            st["wq"] = 1.0 + 0.1 * torch.randn(D, generator=g, device="cuda")
            st["wk"] = 1.0 + 0.1 * torch.randn(D, generator=g, device="cuda")
            st["axes"] = vidax_amd.create_abs_rope3d_axis_freqs(case["T"], case["Y"], case["X"], D, device="cuda")
            st["freqs"] = vidax_amd.create_abs_rope3d_freqs(case["T"], case["Y"], case["X"], D, device="cuda")
        return st
    if kind == "prologue":
        S = case["T"] * case["Y"] * case["X"]
        st["q"], st["k"] = _randn(g, B, S, H * D), _randn(g, B, S, H * D)
        st["wq"] = 1.0 + 0.1 * torch.randn(H * D, generator=g, device="cuda")
        st["wk"] = 1.0 + 0.1 * torch.randn(H * D, generator=g, device="cuda")
        st["freqs"] = vidax_amd.create_rope3d_freqs(case["T"], case["Y"], case["X"], D, device="cuda")
        return st
    S, Sk = case["S"], case.get("Sk", case["S"])
    st["q"], st["k"], st["v"] = _randn(g, B, S, H, D), _randn(g, B, Sk, H, D), _randn(g, B, Sk, H, D)
    if kind == "masked":
        st["valid"] = _valid(case)
    elif kind == "text":
        if case["causal"]:
            st["mask"] = torch.ones((S, S), dtype=torch.bool, device="cuda").tril()[None, None]
        else:
            st["bias"] = torch.randn((1, H, S, S), generator=g, device="cuda")
            st["mask"] = _valid(case)[:, None, None, :]
    elif kind == "cross" and case["kv0"] > 0:
        st["kv_len"] = torch.tensor([case["kv0"], case["kv1"]][:B], dtype=torch.int32, device="cuda")
    elif kind == "key_bias":
        bias = torch.zeros((B, 1, 1, S), device="cuda")
        bias[..., S // 3:S // 3 + case["hole"]] = float("-inf")
        st["bias"] = bias
    return st


# --------------------------------------------------------------------- one pass
def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "masked":
        return vidax_amd.masked_self_attention(st["q"], st["k"], st["v"], key_valid=st["valid"])
    if kind == "text":
        # a T5 layer takes its logits unscaled
        return vidax_amd.dot_product_attention(st["q"], st["k"], st["v"], bias=st.get("bias"), mask=st["mask"],
                                               scale=_scale(case))
    if kind == "cross" and "kv_len" in st:
        return vidax_amd.flash_attention(st["q"], st["k"], st["v"], kv_len=st["kv_len"])
    if kind in ("self", "cross", "key_bias"):
        return vidax_amd.dot_product_attention(st["q"], st["k"], st["v"], bias=st.get("bias"))
    if kind == "na":
        return vidax_amd.neighborhood_attention_3d(st["q"], st["k"], st["v"], st["window"])
    if kind == "na_block":
        k = vidax_amd.na3d_qk_norm_rope(st["k"], st["wk"], st["freqs"])
        return k, vidax_amd.na3d_block_attention(st["q"], k, st["v"], st["window"], st["wq"], st["axes"])
    return (vidax_amd.qk_norm_rope(st["q"], st["wq"], st["freqs"], case["H"]),
            vidax_amd.qk_norm_rope(st["k"], st["wk"], st["freqs"], case["H"]))


def _scale(case):
    # unscaled logits of N(0, 1) inputs would be one-hot at D = 128
    return 1.0 if case["kind"] == "text" and not case["causal"] and case["D"] == 64 else case["D"] ** -0.5


# --------------------------------------------------------------- necessary work
def _keys(case):
    """Valid keys of each batch item."""
    B, S = case["B"], case["S"]
    if case["kind"] in ("masked", "text") and not case.get("causal"):
        return [S - case["pad0"], S - case["pad1"]][:B]
    if case["kind"] == "cross":
        return [case["kv0"] or case["Sk"], case["kv1"] or case["Sk"]][:B]
    if case["kind"] == "key_bias":
        return [S - case["hole"]] * B
    return [S] * B


def work(case):
    kind, B, H, D = case["kind"], case["B"], case["H"], case["D"]
    if kind in ("na", "na_block"):
        n = B * case["T"] * case["Y"] * case["X"] * H
        window = min(case["kt"], case["T"]) * min(case["ky"], case["Y"]) * min(case["kx"], case["X"])
        moved = n * D * 2 * (4 if kind == "na" else 5)  # a block also returns the prepared k
        if kind == "na_block":
            moved += 4 * D * (case["T"] + case["Y"] + case["X"]) + case["T"] * case["Y"] * case["X"] * D * 4
        return {"bytes": moved, "flops": 4.0 * n * window * D}
    if kind == "prologue":
        S = case["T"] * case["Y"] * case["X"]
        return {"bytes": 2 * 2 * B * S * H * D * 2 + S * D * 4 + 2 * H * D * 4, "flops": 2 * 10.0 * B * S * H * D}
    S, keys = case["S"], sum(_keys(case))
    moved = 2 * B * S * H * D * 2 + 2 * keys * H * D * 2
    flops = 4.0 * H * D * S * keys
    if kind == "text":
        moved += S * S if case["causal"] else 4 * H * S * S
        flops *= 0.5 if case["causal"] else 1.0
    if kind in ("masked", "key_bias"):
        moved += B * S * (1 if kind == "masked" else 4)
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    # Measured against exact(), over listed and drawn cases: attention 1.7e-3
    # to 2.4e-3 of the result and at most 0.018 of one value (one rounding of
    # the bf16 output, one of each bf16 probability); the prologue 3.3e-3 and
    # 0.032 (the norm, the weight and the rotation each round to bf16); the
    # block's attention, whose q and k went through that, 5.6e-3 and 0.065.
    # About four times these.
    if case["kind"] == "na_block":
        return {"rel": 2.2e-2, "max": 0.26}
    if case["kind"] == "prologue":
        return {"rel": 1.3e-2, "max": 0.13}
    return {"rel": 1.0e-2, "max": 0.08}


# ------------------------------------------------------------ 64-bit references
def _attend(q, k, v, scale, bias=None):
    """softmax(scale q k^T + bias) v of one head, all (n, D) float64."""
    s = q @ k.t().contiguous()
    s *= scale
    if bias is not None:
        s += bias
    return torch.softmax(s, dim=-1) @ v


def _exact_flash(st):
    case = st["case"]
    kind, B, H = case["kind"], case["B"], case["H"]
    q, k, v = st["q"], st["k"], st["v"]
    S, Sk = q.shape[1], k.shape[1]
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    rows = max(1, (1 << 26) // Sk)
    ninf = torch.tensor(float("-inf"), dtype=torch.float64, device=q.device)
    for b in range(B):
        keep = torch.ones(Sk, dtype=torch.bool, device=q.device)
        if kind == "masked":
            keep = st["valid"][b]
        elif kind == "text" and not case["causal"]:
            keep = st["mask"][b, 0, 0]
        elif kind == "cross" and "kv_len" in st:
            keep = torch.arange(Sk, device=q.device) < st["kv_len"][b]
        elif kind == "key_bias":
            keep = st["bias"][b, 0, 0] == 0
        idx = keep.nonzero()[:, 0]
        for h in range(H):
            kh, vh = k[b, idx, h].double(), v[b, idx, h].double()
            for r in range(0, S, rows):
                bias = None
                if kind == "text":
                    if case["causal"]:
                        bias = torch.where(st["mask"][0, 0, r:r + rows], 0.0, ninf)
                    else:
                        bias = st["bias"][0, h, r:r + rows][:, idx].double()
                out[b, r:r + rows, h] = _attend(q[b, r:r + rows, h].double(), kh, vh, _scale(case), bias)
    return out.reshape(B, S, -1) if kind == "masked" else out


def _axis_angles(n, freqs):
    return torch.arange(n, dtype=torch.float64, device="cuda")[:, None] * freqs[None, :]


def _angles(case, pairs):
    """(T*Y*X, D/2) rotation angles; pairs: pairs of the t, y and x axes, each
    with frequencies 10000^(-j / pairs)."""
    T, Y, X = case["T"], case["Y"], case["X"]
    a = []
    for n, p, view in ((T, pairs[0], (T, 1, 1, -1)), (Y, pairs[1], (1, Y, 1, -1)), (X, pairs[2], (1, 1, X, -1))):
        f = 10000.0 ** (-torch.arange(p, dtype=torch.float64, device="cuda") / p)
        a.append(_axis_angles(n, f).reshape(view).expand(T, Y, X, p))
    return torch.cat(a, dim=-1).reshape(T * Y * X, -1)


def _rotate(x, ang):
    """x (B, S, H, D) float64, pairs (2j, 2j + 1) turned by ang (S, D/2)."""
    c, s = ang.cos()[None, :, None, :], ang.sin()[None, :, None, :]
    x1, x2 = x[..., 0::2], x[..., 1::2]
    return torch.stack([x1 * c - x2 * s, x2 * c + x1 * s], dim=-1).flatten(-2)


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w


def _exact_na(case, q, k, v, window):
    """Row by row of the (t, y) grid: the query row's W tokens against the
    window's kt x ky key rows, the x window as a mask."""
    T, Y, X, H, D = case["T"], case["Y"], case["X"], case["H"], case["D"]
    kt, ky, kx = min(window[0], T), min(window[1], Y), min(window[2], X)

    def start(i, n, w):
        return min(max(i - w // 2, 0), n - w)

    xs = torch.tensor([start(i, X, kx) for i in range(X)], device="cuda")
    pos = torch.arange(X, device="cuda")
    out_x = (pos[None, :] < xs[:, None]) | (pos[None, :] >= (xs + kx)[:, None])  # (query, key)
    q, k, v = (x[0].permute(3, 0, 1, 2, 4).contiguous() for x in (q, k, v))      # (H, T, Y, X, D)
    out = torch.empty_like(q)
    for t in range(T):
        t0 = start(t, T, kt)
        for y in range(Y):
            y0 = start(y, Y, ky)
            kb = k[:, t0:t0 + kt, y0:y0 + ky].reshape(H, -1, D)
            vb = v[:, t0:t0 + kt, y0:y0 + ky].reshape(H, -1, D).contiguous()
            s = torch.bmm(q[:, t, y].contiguous(), kb.transpose(1, 2).contiguous())
            s = s.reshape(H, X, kt * ky, X).masked_fill_(out_x[None, :, None, :], float("-inf")).reshape(H, X, -1)
            out[:, t, y] = torch.bmm(torch.softmax(s, dim=-1), vb)
    return out.permute(1, 2, 3, 0, 4)[None].contiguous()


def exact(case, seed):
    kind, D = case["kind"], case["D"]
    if kind in ("na", "na_block"):
        n = case["T"] * case["Y"] * case["X"] * case["H"]
        if n * D * min(case["kt"], case["T"]) * min(case["ky"], case["Y"]) * case["X"] > 4e13:
            return None
    elif work(case)["flops"] > 4e13:
        return None
    st = prepare(case, seed)
    if kind == "prologue":
        p = D // 2 // 3
        ang = _angles(case, (D // 2 - 2 * p, p, p))
        outs = []
        for x, w in ((st["q"], st["wq"]), (st["k"], st["wk"])):
            y = _rms(x.double(), w.double()).reshape(x.shape[0], x.shape[1], case["H"], D)
            outs.append(_rotate(y, ang))
        return tuple(outs)
    if kind == "na":
        return _exact_na(case, st["q"].double(), st["k"].double(), st["v"].double(), st["window"])
    if kind == "na_block":
        d_t = D // 4 // 2 * 2
        d_t -= 2 if (D - d_t) // 2 % 2 else 0
        ang = _angles(case, (d_t // 2, (D - d_t) // 4, (D - d_t) // 4))
        shape = st["q"].shape
        flat = (shape[0], -1, case["H"], D)
        q = _rotate((_rms(st["q"].double(), st["wq"].double()) * D ** -0.5).reshape(flat), ang).reshape(shape)
        k = _rotate(_rms(st["k"].double(), st["wk"].double()).reshape(flat), ang).reshape(shape)
        return k, _exact_na(case, q, k, st["v"].double(), st["window"])
    return _exact_flash(st)
