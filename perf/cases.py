"""Performance cases of the Evoformer path: what a ColabFold-style program calls this library for.

A case is one call, or the few calls of one layer, through ``colabfold_legacy_kernels.ops``:

  pair_block   LN + both gated projections, the pair bias and the attention of one pair block
  attn_train   triangle attention forward (with the logsumexp) and backward
  msa_train    MSA row attention with its output gate through autograd, forward and backward
  attn_infer   triangle attention forward
  gated_infer  triangle attention forward, then the output gate
  extra_msa    extra-MSA row attention forward (head dim 8) on the [N,S,H,D] layout
  ln_gdp       LayerNorm + both gated projections of the triangle multiplication, forward
  ln_gdp_bwd   its backward
  layer_norm   LayerNorm forward and backward
  tri_mult     the whole triangle multiplication, outgoing or incoming

Residue counts are those of proteins, so most of them are no multiple of anything; the round ones
are training crops and padded buckets. ``exact`` restates every case in float64 with plain torch.
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "colabfold-legacy-kernels_amd"))

from colabfold_legacy_kernels import ops  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_EPS = 1e-5
_DEVICE = "cuda"


def listed():
    return [
        # One pair block of a 64-residue chain: four short calls, where launches and latency count.
        {"name": "pair_block_64", "kind": "pair_block", "dtype": "bf16", "r": 64, "c": 128,
         "h": 4, "d": 32},
        # Triangle attention of a 384-residue training crop, its last tenth padding.
        {"name": "attn_train_384", "kind": "attn_train", "dtype": "bf16", "r": 384, "h": 4,
         "d": 32, "tail": 0.1},
        # The same step on a whole chain of 203 residues, nothing rounded up, in float16.
        {"name": "attn_train_203", "kind": "attn_train", "dtype": "f16", "r": 203, "h": 4,
         "d": 32, "tail": 0.0},
        # MSA row attention in training: 512 sequences, a fifth of them padding, gated output.
        {"name": "msa_train_512x256", "kind": "msa_train", "dtype": "bf16", "n": 512, "r": 256,
         "h": 8, "d": 32, "c": 256, "pad_rows": 0.2},
        # Prediction of a 757-residue chain: triangle attention forward on unpadded rows.
        {"name": "attn_infer_757", "kind": "attn_infer", "dtype": "bf16", "r": 757, "h": 4,
         "d": 32, "tail": 0.0},
        # Prediction of a large complex in a 1024 bucket, the output gated.
        {"name": "gated_infer_1024", "kind": "gated_infer", "dtype": "bf16", "r": 1024, "h": 4,
         "d": 32, "c": 128, "tail": 0.15},
        # Extra-MSA row attention (8 heads of 8): 1024 sequences of 300 residues.
        {"name": "extra_msa_1024x300", "kind": "extra_msa", "dtype": "f16", "n": 1024, "r": 300,
         "h": 8, "d": 8, "tail": 0.0},
        # LayerNorm + gated dual projections of a 512-residue pair representation, forward.
        {"name": "ln_gdp_512", "kind": "ln_gdp", "dtype": "bf16", "r": 512, "c": 128, "n": 128},
        # Their backward on a chain of 301 residues.
        {"name": "ln_gdp_bwd_301", "kind": "ln_gdp_bwd", "dtype": "bf16", "r": 301, "c": 128,
         "n": 128},
        # LayerNorm forward and backward over a 512-residue pair representation.
        {"name": "layer_norm_512", "kind": "layer_norm", "dtype": "bf16", "m": 512 * 512,
         "c": 128},
        # Triangle multiplication, outgoing, at a round size and incoming at an odd one.
        {"name": "tri_mult_512", "kind": "tri_mult", "dtype": "bf16", "r": 512, "c": 128,
         "outgoing": True},
        {"name": "tri_mult_389", "kind": "tri_mult", "dtype": "f16", "r": 389, "c": 128,
         "outgoing": False},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    """One more case of the listed kinds: sizes spread over the logarithm of their range."""
    kind = rng.choice(["pair_block", "attn_train", "msa_train", "attn_infer", "gated_infer",
                       "extra_msa", "ln_gdp", "ln_gdp_bwd", "layer_norm", "tri_mult"])
    case = {"kind": kind, "dtype": rng.choice(["bf16", "f16"])}
    heads = rng.choice([(4, 32), (4, 32), (4, 16)])  # pair stack, or the template stack
    tail = rng.choice([0.0, 0.0, 0.1, 0.15, 0.3])
    if kind == "pair_block":
        case.update(r=_log_int(rng, 16, 128), c=128, h=4, d=32)
    elif kind == "attn_train":
        case.update(r=_log_int(rng, 32, 512), h=heads[0], d=heads[1], tail=tail)
    elif kind == "msa_train":
        case.update(n=_log_int(rng, 32, 512), r=_log_int(rng, 48, 320), h=8, d=32, c=256,
                    pad_rows=rng.choice([0.0, 0.2]))
    elif kind == "attn_infer":
        case.update(r=_log_int(rng, 32, 768), h=heads[0], d=heads[1], tail=tail)
    elif kind == "gated_infer":
        case.update(r=_log_int(rng, 64, 1024), h=4, d=32, c=128, tail=tail)
    elif kind == "extra_msa":
        case.update(n=_log_int(rng, 128, 1024), r=_log_int(rng, 48, 384), h=8, d=8, tail=tail)
    elif kind in ("ln_gdp", "ln_gdp_bwd"):
        width = rng.choice([128, 128, 64])
        case.update(r=_log_int(rng, 32, 512), c=width, n=width)
    elif kind == "layer_norm":
        # Pair (128), template (64), MSA (256) and single (384) widths; float32 as well.
        case.update(dtype=rng.choice(["bf16", "f16", "f32"]), m=_log_int(rng, 64, 512 * 512),
                    c=rng.choice([64, 128, 256, 384]))
        case["m"] = max(64, case["m"] * 128 // case["c"] if case["c"] > 128 else case["m"])
    else:
        case.update(r=_log_int(rng, 32, 640), c=rng.choice([128, 128, 64]),
                    outgoing=rng.choice([True, False]))
    return case


# ---- inputs ----------------------------------------------------------------------------------

class _Rand:
    """Seeded normal draws on the device, rounded to the case's type."""

    def __init__(self, seed, dtype):
        self.g = torch.Generator(device=_DEVICE)
        self.g.manual_seed(int(seed))
        self.dtype = dtype

    def n(self, *shape, std=1.0, mean=0.0, dtype=None):
        t = torch.randn(shape, generator=self.g, device=_DEVICE, dtype=torch.float32)
        return t.mul_(std).add_(mean).to(dtype or self.dtype)

    def keep(self, *shape, p):
        return torch.rand(shape, generator=self.g, device=_DEVICE) < p


def _ln_params(rand, c):
    f32 = torch.float32
    return rand.n(c, std=0.3, mean=1.0, dtype=f32), rand.n(c, std=0.3, dtype=f32)


def _branch(rand, c, n):
    """(wp, bp, wg, bg) of one gated dual projection."""
    std = 1.0 / math.sqrt(c)
    return (rand.n(c, n, std=std), rand.n(n, std=0.1), rand.n(c, n, std=std),
            rand.n(n, std=0.1))


def _attention(rand, n, r, h, d, tail=0.0, pad_rows=0.0, nshd=False):
    shape = (n, r, h, d) if nshd else (n, h, r, d)
    kmask = torch.ones((n, r), dtype=torch.uint8, device=_DEVICE)
    absent = int(round(tail * r))
    if absent:
        kmask[:, r - absent:] = 0
    rows = int(round(pad_rows * n))
    if rows:
        kmask[torch.randperm(n, generator=rand.g, device=_DEVICE)[:rows]] = 0
    return {"q": rand.n(*shape), "k": rand.n(*shape), "v": rand.n(*shape),
            "bias": rand.n(h, r, r), "kmask": kmask}


def prepare(case, seed):
    kind, dtype = case["kind"], _DTYPES[case["dtype"]]
    rand = _Rand(seed, dtype)
    s = {"case": case}
    if kind == "pair_block":
        r, c, h, d = case["r"], case["c"], case["h"], case["d"]
        s.update(_attention(rand, r, r, h, d))
        s.update(z=rand.n(r, r, c), ln=_ln_params(rand, c), a=_branch(rand, c, c),
                 b=_branch(rand, c, c), wb=rand.n(c, h, std=1.0 / math.sqrt(c)),
                 mask=torch.ones((r, r), device=_DEVICE, dtype=dtype))
        del s["bias"]
    elif kind in ("attn_train", "attn_infer"):
        s.update(_attention(rand, case["r"], case["r"], case["h"], case["d"], case["tail"]))
        if kind == "attn_train":
            s["dout"] = rand.n(case["r"], case["h"], case["r"], case["d"])
    elif kind in ("msa_train", "gated_infer"):
        n, r, h, d, c = case.get("n", case["r"]), case["r"], case["h"], case["d"], case["c"]
        s.update(_attention(rand, n, r, h, d, case.get("tail", 0.0), case.get("pad_rows", 0.0)))
        s.update(x=rand.n(n, r, c), wg=rand.n(c, h * d, std=1.0 / math.sqrt(c)),
                 bg=rand.n(h * d, std=0.1))
        if kind == "msa_train":
            s["dout"] = rand.n(n, r, h * d)
            for name in ("q", "k", "v", "bias", "x", "wg", "bg"):
                s[name].requires_grad_(True)
    elif kind == "extra_msa":
        s.update(_attention(rand, case["n"], case["r"], case["h"], case["d"], case["tail"],
                            nshd=True))
    elif kind in ("ln_gdp", "ln_gdp_bwd"):
        r, c, n = case["r"], case["c"], case["n"]
        s.update(z=rand.n(r, r, c), ln=_ln_params(rand, c), a=_branch(rand, c, n),
                 b=_branch(rand, c, n), mask=rand.keep(r, r, p=0.95).to(dtype))
        if kind == "ln_gdp_bwd":
            s.update(da=rand.n(r, r, n), db=rand.n(r, r, n))
    elif kind == "layer_norm":
        s.update(x=rand.n(case["m"], case["c"]), ln=_ln_params(rand, case["c"]),
                 dy=rand.n(case["m"], case["c"]))
    else:
        r, c = case["r"], case["c"]
        s.update(z=rand.n(r, r, c), mask=rand.keep(r, r, p=0.95).to(dtype),
                 ln=_ln_params(rand, c), ln_center=_ln_params(rand, c),
                 w=[rand.n(c, c, std=1.0 / math.sqrt(c)) for _ in range(6)],
                 wb=[rand.n(c, std=0.1) for _ in range(6)])
    return s


# ---- one pass --------------------------------------------------------------------------------

def run(s):
    kind = s["case"]["kind"]
    if kind == "pair_block":
        a, b = ops.ln_gated_dual_proj(s["z"], *s["ln"], s["a"], s["b"], s["mask"], _EPS)
        bias = ops.ln_pair_bias(s["z"], *s["ln"], s["wb"], _EPS)
        return [a, b, bias, ops.attention(s["q"], s["k"], s["v"], bias, s["kmask"])]
    if kind == "attn_train":
        args = (s["q"], s["k"], s["v"], s["bias"], s["kmask"])
        out, lse = ops.attention_fwd(*args)
        return [out, lse, *ops.attention_bwd(*args, out, s["dout"], lse)]
    if kind == "attn_infer":
        return ops.attention(s["q"], s["k"], s["v"], s["bias"], s["kmask"])
    if kind == "msa_train":
        leaves = tuple(s[name] for name in ("q", "k", "v", "bias", "x", "wg", "bg"))
        out = ops.GatedAttentionFunction.apply(*leaves[:4], s["kmask"], *leaves[4:],
                                               1.0 / math.sqrt(s["case"]["d"]))
        return [out.detach(), *torch.autograd.grad(out, leaves, s["dout"])]
    if kind == "gated_infer":
        out = ops.attention(s["q"], s["k"], s["v"], s["bias"], s["kmask"])
        return ops.attention_gate(out, s["x"], s["wg"], s["bg"])
    if kind == "extra_msa":
        return ops.attention_nshd(s["q"], s["k"], s["v"], s["bias"], s["kmask"])[0]
    if kind == "ln_gdp":
        return list(ops.ln_gated_dual_proj(s["z"], *s["ln"], s["a"], s["b"], s["mask"], _EPS))
    if kind == "ln_gdp_bwd":
        dz, dscale, doffset, ga, gb = ops.ln_gated_dual_proj_bwd(
            s["z"], *s["ln"], s["a"], s["b"], s["mask"], s["da"], s["db"], _EPS)
        return [dz, dscale, doffset, *ga, *gb]
    if kind == "layer_norm":
        y = ops.layer_norm(s["x"], *s["ln"], _EPS)
        return [y, *ops.layer_norm_bwd(s["x"], s["ln"][0], s["dy"], _EPS)]
    return ops.triangle_multiply(s["z"], s["mask"], s["ln"], s["w"], s["wb"], s["ln_center"],
                                 s["case"]["outgoing"], _EPS)


# ---- what a pass cannot do without -----------------------------------------------------------

def work(case):
    kind, r = case["kind"], case.get("r", 0)
    e = 4 if case["dtype"] == "f32" else 2
    if kind in ("pair_block", "attn_train", "msa_train", "attn_infer", "gated_infer",
                "extra_msa"):
        n, h, d, c = case.get("n", r), case["h"], case["d"], case.get("c", 0)
        qkvo = n * h * r * d * e  # one of q, k, v, out and their gradients
        scores = n * h * r * r * d
        shared = h * r * r * e + n * r  # the bias and the mask
        gate_b = n * r * c * e + (c + 1) * h * d * e
        gate_f = 2 * n * r * c * h * d
        if kind in ("attn_infer", "extra_msa"):
            return {"bytes": 4 * qkvo + shared, "flops": 4 * scores}
        if kind == "gated_infer":
            return {"bytes": 4 * qkvo + shared + gate_b, "flops": 4 * scores + gate_f}
        if kind == "attn_train":
            # q, k, v, dout in; out, lse, dq, dk, dv and the float32 dbias out.
            return {"bytes": 8 * qkvo + shared + 4 * n * h * r + 4 * h * r * r,
                    "flops": 12 * scores}
        if kind == "msa_train":
            return {"bytes": 8 * qkvo + shared + h * r * r * e + 2 * gate_b,
                    "flops": 12 * scores + 3 * gate_f}
        pair = r * r * c * e
        weights = (4 * c * c + c * h) * e
        return {"bytes": 3 * pair + r * r * (1 + h) * e + weights + 4 * qkvo + n * r,
                "flops": 8 * r * r * c * c + 2 * r * r * c * h + 4 * scores}
    if kind in ("ln_gdp", "ln_gdp_bwd"):
        c, n = case["c"], case["n"]
        m = r * r
        weights = 4 * (c * n + n) * e
        if kind == "ln_gdp":
            return {"bytes": m * (c + 2 * n + 1) * e + weights + 8 * c, "flops": 8 * m * c * n}
        # z, da, db, mask in, dz out, weights in and their float32 gradients out; the recomputed
        # projections, dy and the weight gradients.
        return {"bytes": m * (2 * c + 2 * n + 1) * e + weights + 2 * weights + 16 * c,
                "flops": 24 * m * c * n}
    if kind == "layer_norm":
        m, c = case["m"], case["c"]
        return {"bytes": 4 * m * c * e + 16 * c, "flops": 20 * m * c}
    c = case["c"]
    return {"bytes": 2 * r * r * c * e + r * r * e + 6 * (c * c + c) * e + 16 * c,
            "flops": 2 * r ** 3 * c + 12 * r * r * c * c}


# Relative errors of another correct implementation at the same precision, about four times what
# this library shows against float64: 16-bit results of float32 sums (the rounding of the result
# and of the probabilities, projections or normalised rows that enter the matrix products), and
# float32 sums of them.
_REL = {"pair_block": 1.2e-2, "attn_train": 1e-2, "msa_train": 1.2e-2, "attn_infer": 1e-2,
        "gated_infer": 1.2e-2, "extra_msa": 1e-2, "ln_gdp": 1.2e-2, "ln_gdp_bwd": 1.4e-2,
        "layer_norm": 7e-3, "tri_mult": 1.6e-2}


def tolerance(case):
    if case["dtype"] == "f32":
        return {"rel": 2e-6}
    rel = _REL[case["kind"]]
    # float16 keeps three bits more than bfloat16.
    return {"rel": rel / 8 if case["dtype"] == "f16" else rel}


# ---- the same in float64 ---------------------------------------------------------------------

def _attention64(q, k, v, bias, kmask, scale, dout=None):
    """o, lse and, given dout, dq, dk, dv, dbias of attention with the additive mask convention:
    an absent key has the logit -1e9 and the gradient of every key is P * (dP - D); in a row with
    no present key the softmax is uniform (logit 0, lse ln Sk). A few rows at a time."""
    n, h, sq, _ = q.shape
    sk = k.shape[2]
    step = max(1, (1 << 27) // (h * sq * sk))
    o, lse = [], []
    grads = [[], [], []]
    dbias = torch.zeros((h, sq, sk), dtype=torch.float64, device=q.device)
    for i in range(0, n, step):
        qd, kd, vd = (t[i:i + step].double() for t in (q, k, v))
        present = kmask[i:i + step].bool()
        fill = torch.where(present.any(1), -1e9, 0.0).double()[:, None, None, None]
        s = torch.matmul(qd, kd.transpose(-1, -2).contiguous()) * scale + bias.double()
        s = torch.where(present[:, None, None, :], s, fill)
        li = torch.logsumexp(s, -1)
        p = torch.exp(s - li[..., None])
        oi = torch.matmul(p, vd)
        o.append(oi)
        lse.append(li)
        if dout is not None:
            dd = dout[i:i + step].double()
            ds = torch.matmul(dd, vd.transpose(-1, -2).contiguous())
            ds = p * (ds - (dd * oi).sum(-1, keepdim=True))
            dbias += ds.sum(0)
            grads[0].append(scale * torch.matmul(ds, kd))
            grads[1].append(scale * torch.matmul(ds.transpose(-1, -2).contiguous(), qd))
            grads[2].append(torch.matmul(p.transpose(-1, -2).contiguous(), dd))
    return (torch.cat(o), torch.cat(lse), *(torch.cat(g) if g else None for g in grads), dbias)


def _ln64(x, scale, offset):
    mean = x.mean(-1, keepdim=True)
    var = (x - mean).square().mean(-1, keepdim=True)
    return (x - mean) * torch.rsqrt(var + _EPS) * scale + offset


def _gdp64(y, branch, mask):
    wp, bp, wg, bg = branch
    return mask[..., None] * (y @ wp + bp) * torch.sigmoid(y @ wg + bg)


def _d(ts):
    return tuple(t.detach().double() for t in ts)


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind in ("pair_block", "attn_train", "msa_train", "attn_infer", "gated_infer",
                "extra_msa"):
        q, k, v = (s[name].detach() for name in ("q", "k", "v"))
        scale = 1.0 / math.sqrt(case["d"])
        if kind == "pair_block":
            y = _ln64(s["z"].double(), *_d(s["ln"]))
            bias = (y @ s["wb"].double()).permute(2, 0, 1).contiguous()
            mask = s["mask"].double()
            return [_gdp64(y, _d(s["a"]), mask), _gdp64(y, _d(s["b"]), mask), bias,
                    _attention64(q, k, v, bias, s["kmask"], scale)[0]]
        bias = s["bias"].detach()
        if kind == "attn_infer":
            return _attention64(q, k, v, bias, s["kmask"], scale)[0]
        if kind == "extra_msa":
            q, k, v = (t.transpose(1, 2) for t in (q, k, v))
            return _attention64(q, k, v, bias, s["kmask"], scale)[0].transpose(1, 2).contiguous()
        if kind == "attn_train":
            return list(_attention64(q, k, v, bias, s["kmask"], scale, s["dout"]))
        x, wg, bg = _d((s["x"], s["wg"], s["bg"]))
        n, r, h, d = q.shape[0], case["r"], case["h"], case["d"]
        gate = torch.sigmoid(x @ wg + bg)
        if kind == "gated_infer":
            o = _attention64(q, k, v, bias, s["kmask"], scale)[0]
            return o.transpose(1, 2).reshape(n, r, h * d) * gate
        dg = s["dout"].double()
        do = (dg * gate).view(n, r, h, d).transpose(1, 2)
        o, _, dq, dk, dv, dbias = _attention64(q, k, v, bias, s["kmask"], scale, do)
        o = o.transpose(1, 2).reshape(n, r, h * d)
        dl = (dg * o * gate * (1 - gate)).view(n * r, h * d)
        c = case["c"]
        return [o * gate, dq, dk, dv, dbias, (dl @ wg.t().contiguous()).view(n, r, c),
                x.view(n * r, c).t().contiguous() @ dl, dl.sum(0)]
    if kind in ("ln_gdp", "ln_gdp_bwd"):
        z, scale, offset, mask = _d((s["z"], *s["ln"], s["mask"]))
        a, b = _d(s["a"]), _d(s["b"])
        if kind == "ln_gdp":
            y = _ln64(z, scale, offset)
            return [_gdp64(y, a, mask), _gdp64(y, b, mask)]
        leaves = [t.requires_grad_(True) for t in (z, scale, offset, *a, *b)]
        y = _ln64(z, scale, offset)
        outs = (_gdp64(y, a, mask), _gdp64(y, b, mask))
        return list(torch.autograd.grad(outs, leaves, _d((s["da"], s["db"]))))
    if kind == "layer_norm":
        leaves = [t.requires_grad_(True) for t in _d((s["x"], *s["ln"]))]
        y = _ln64(*leaves)
        return [y.detach(), *torch.autograd.grad(y, leaves, s["dy"].double())]
    z, mask = _d((s["z"], s["mask"]))
    w, wb = _d(s["w"]), _d(s["wb"])
    y = _ln64(z, *_d(s["ln"]))
    left = _gdp64(y, (w[0], wb[0], w[2], wb[2]), mask).permute(2, 0, 1).contiguous()
    right = _gdp64(y, (w[1], wb[1], w[3], wb[3]), mask).permute(2, 0, 1).contiguous()
    if case["outgoing"]:
        x = torch.matmul(left, right.transpose(1, 2).contiguous())
    else:
        x = torch.matmul(right.transpose(1, 2).contiguous(), left)
    x = _ln64(x.permute(1, 2, 0).contiguous(), *_d(s["ln_center"]))
    return (x @ w[4] + wb[4]) * torch.sigmoid(y @ w[5] + wb[5])
