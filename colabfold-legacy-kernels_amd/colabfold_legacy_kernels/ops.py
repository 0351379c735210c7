"""PyTorch front end of the gfx950 kernels: allocate outputs, pass pointers to the C ABI.

Each function mirrors one XLA FFI target of the reference -- the same operands in the same order,
the same attributes, the same errors -- with torch tensors on a ROCm device in place of XLA
buffers:

  attention(q, k, v, bias, kmask, scale, block_q, block_k)   VoltaMma   (cuda/volta_mma_attn.cu:338-351)
  layer_norm(x, scale, offset, eps)                          VoltaLayerNorm (cuda/volta_ops.cu:87-95)
  gated_dual_proj(x, wp, bp, wg, bg, mask)                   VoltaGdp   (cuda/volta_ops.cu:254-265)

and the targets the reference lacks: attention_fwd (also returns the logsumexp), attention_bwd,
layer_norm_bwd and ln_gated_dual_proj. An invalid call raises InvalidArgument (a ValueError), as
the reference handlers return ffi::Error::InvalidArgument; a launch failure raises InternalError.

Torch is used only for device memory and the current stream; all arithmetic runs in the HIP
library, and a missing library raises FileNotFoundError (there is no fallback path).
"""

import ctypes
import math

import torch

from . import _native

__all__ = [
    "ClkError", "InvalidArgument", "InternalError",
    "attention", "attention_fwd", "attention_bwd",
    "attention_gate", "attention_gate_bwd", "attention_gated", "attention_gated_fwd",
    "layer_norm", "layer_norm_bwd",
    "gated_dual_proj", "ln_gated_dual_proj",
    "AttentionFunction", "GatedAttentionFunction", "LayerNormFunction",
]


class ClkError(RuntimeError):
    """A non-OK status from the library; ``code`` is the clk_status value."""

    def __init__(self, code, message):
        super().__init__(message)
        self.code = code


class InvalidArgument(ClkError, ValueError):
    pass


class InternalError(ClkError):
    pass


_DTYPES = {torch.float16: _native.F16, torch.bfloat16: _native.BF16,
           torch.float32: _native.F32}


def _check(status):
    if status == _native.OK:
        return
    msg = _native.last_error()
    if status == _native.INVALID_ARGUMENT:
        raise InvalidArgument(status, msg)
    raise InternalError(status, msg)


def _ptr(t):
    return None if t is None else t.data_ptr()


def _dtype_code(t, allowed, what):
    code = _DTYPES.get(t.dtype)
    if code is None or code not in allowed:
        raise InvalidArgument(_native.INVALID_ARGUMENT,
                              "%s: dtype %s not supported" % (what, t.dtype))
    return code


def _require(tensors, what):
    """The index of the one ROCm device that holds every given (contiguous) tensor."""
    index = None
    for name, t in tensors:
        if t is None:
            continue
        if not isinstance(t, torch.Tensor) or not t.is_cuda:
            raise InvalidArgument(_native.INVALID_ARGUMENT,
                                  "%s: %s must be a tensor on a ROCm device" % (what, name))
        if not t.is_contiguous():
            raise InvalidArgument(_native.INVALID_ARGUMENT, "%s: %s must be contiguous" % (what, name))
        if index is None:
            index = t.get_device()
        elif t.get_device() != index:
            raise InvalidArgument(_native.INVALID_ARGUMENT,
                                  "%s: all operands must be on one device" % what)
    return index


# The raw handle of a device's current stream, without building a Stream object where torch has
# the direct call (1.8 us against 0.1).
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
if _raw_stream is None:
    def _raw_stream(index):
        return torch.cuda.current_stream(index).cuda_stream


def _launch(index, fn, *args):
    """fn(stream, *args) on device `index`, its current stream first; raises on a bad status. The
    device is switched only when it is not the current one (a context costs 1.3 us)."""
    if torch.cuda.current_device() == index:
        status = fn(_raw_stream(index), *args)
    else:
        with torch.cuda.device(index):
            status = fn(_raw_stream(index), *args)
    if status != _native.OK:
        _check(status)


def _fail(what, msg):
    raise InvalidArgument(_native.INVALID_ARGUMENT, "%s: %s" % (what, msg))


def _all_dtype(dtype, tensors):
    for t in tensors:
        if t.dtype != dtype:
            return False
    return True


def _shape_check(cond, what, msg):
    if not cond:
        _fail(what, msg)


def _workspace(t, nbytes):
    return t.new_empty(max(nbytes, 1), dtype=torch.uint8)


def _attn_dims(q, k, v, bias, kmask, what, nshd=False):
    """(n, h, sq, sk, d) of [N,H,S,D] operands, or of [N,S,H,D] ones with nshd."""
    qs, ks = q.shape, k.shape
    if len(qs) != 4:
        _fail(what, "q must be [N,H,S,D]")
    n, h, sq, d = qs
    if nshd:
        h, sq = sq, h
    if len(ks) != 4:
        _fail(what, "k must be [N,H,Sk,D]")
    kh, sk = (ks[2], ks[1]) if nshd else (ks[1], ks[2])
    if ks[0] != n or kh != h or ks[3] != d:
        _fail(what, "k must be [N,H,Sk,D]")
    if v.shape != ks:
        _fail(what, "v must have the shape of k")
    if bias.shape != (h, sq, sk):
        _fail(what, "bias must be [H,Sq,Sk]")
    dtype = q.dtype
    if k.dtype != dtype or v.dtype != dtype or bias.dtype != dtype:
        _fail(what, "q, k, v and bias must share one dtype")
    if kmask is not None and (kmask.shape != (n, sk) or kmask.dtype != torch.uint8):
        _fail(what, "kmask must be uint8 [N,Sk]")
    return n, h, sq, sk, d


def _attention_call(q, k, v, bias, kmask, scale, block_q, block_k, want_lse, what):
    index = _require([("q", q), ("k", k), ("v", v), ("bias", bias), ("kmask", kmask)], what)
    n, h, sq, sk, d = _attn_dims(q, k, v, bias, kmask, what)
    code = _dtype_code(q, (_native.F16, _native.BF16), what)
    if scale is None:
        scale = 1.0 / math.sqrt(d)
    out = torch.empty_like(q)
    lse = q.new_empty((n, h, sq), dtype=torch.float32) if want_lse else None
    lib = _native.lib()
    _launch(index, lib.clk_attention_fwd, code, q.data_ptr(), k.data_ptr(), v.data_ptr(),
            bias.data_ptr(), _ptr(kmask), out.data_ptr(), _ptr(lse), n, h, sq, sk, d, float(scale),
            int(block_q), int(block_k))
    return out, lse


def attention(q, k, v, bias, kmask=None, scale=None, block_q=64, block_k=64):
    """softmax(scale*q.k^T + bias, masked keys -> -1e9) . v for q [N,H,Sq,D], k/v [N,H,Sk,D],
    bias [H,Sq,Sk], kmask uint8 [N,Sk]. block_q/block_k are accepted as hints."""
    out, _ = _attention_call(q, k, v, bias, kmask, scale, block_q, block_k, False, "attention")
    return out


def attention_fwd(q, k, v, bias, kmask=None, scale=None):
    """(out, lse): the forward plus the float32 natural-log logsumexp [N,H,Sq] per query."""
    return _attention_call(q, k, v, bias, kmask, scale, 64, 64, True, "attention_fwd")


def attention_nshd(q, k, v, bias, kmask=None, scale=None, want_lse=False):
    """The forward on AlphaFold's [N,S,H,D] layout: q [N,Sq,H,D], k/v [N,Sk,H,D], bias
    [H,Sq,Sk], kmask uint8 [N,Sk]; returns (out [N,Sq,H,D], lse [N,H,Sq] or None), bit-identical
    to attention_fwd on the [N,H,S,D] transposes."""
    what = "attention_nshd"
    index = _require([("q", q), ("k", k), ("v", v), ("bias", bias), ("kmask", kmask)], what)
    _shape_check(q.dim() == 4 and k.dim() == 4, what, "q and k must be [N,S,H,D]")
    n, h, sq, sk, d = _attn_dims(q, k, v, bias, kmask, what, nshd=True)
    code = _dtype_code(q, (_native.F16, _native.BF16), what)
    if scale is None:
        scale = 1.0 / math.sqrt(d)
    out = torch.empty_like(q)
    lse = q.new_empty((n, h, sq), dtype=torch.float32) if want_lse else None
    lib = _native.lib()
    _launch(index, lib.clk_attention_fwd_nshd, code, q.data_ptr(), k.data_ptr(), v.data_ptr(),
            bias.data_ptr(), _ptr(kmask), out.data_ptr(), _ptr(lse), n, h, sq, sk, d, float(scale))
    return out, lse


def attention_bwd(q, k, v, bias, kmask, out, dout, lse, scale=None):
    """(dq, dk, dv, dbias) with dbias [H,Sq,Sk] float32 summed over the N rows."""
    what = "attention_bwd"
    index = _require([("q", q), ("k", k), ("v", v), ("bias", bias), ("kmask", kmask),
                      ("out", out), ("dout", dout), ("lse", lse)], what)
    n, h, sq, sk, d = _attn_dims(q, k, v, bias, kmask, what)
    code = _dtype_code(q, (_native.F16, _native.BF16), what)
    _shape_check(out.shape == q.shape and out.dtype == q.dtype, what,
                 "out must match q")
    _shape_check(dout.shape == q.shape and dout.dtype == q.dtype, what,
                 "dout must match q")
    _shape_check(lse.shape == (n, h, sq) and lse.dtype == torch.float32, what,
                 "lse must be float32 [N,H,Sq]")
    if scale is None:
        scale = 1.0 / math.sqrt(d)
    lib = _native.lib()
    ws_bytes = lib.clk_attention_bwd_workspace_size(n, h, sq, sk, d)
    ws = _workspace(q, ws_bytes)
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    dbias = q.new_empty((h, sq, sk), dtype=torch.float32)
    _launch(index, lib.clk_attention_bwd, code, q.data_ptr(), k.data_ptr(), v.data_ptr(),
            bias.data_ptr(), _ptr(kmask), out.data_ptr(), dout.data_ptr(), lse.data_ptr(),
            dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), dbias.data_ptr(), ws.data_ptr(), ws_bytes,
            n, h, sq, sk, d, float(scale))
    return dq, dk, dv, dbias


def attention_bwd_nshd(q, k, v, bias, kmask, out, dout, lse, scale=None):
    """attention_bwd on AlphaFold's [N,S,H,D] layout: q, out, dout [N,Sq,H,D], k, v [N,Sk,H,D],
    lse [N,H,Sq]; returns (dq, dk, dv) in the layout of q, k, v and dbias [H,Sq,Sk] float32,
    bit-identical to attention_bwd on the [N,H,S,D] transposes."""
    what = "attention_bwd_nshd"
    index = _require([("q", q), ("k", k), ("v", v), ("bias", bias), ("kmask", kmask),
                      ("out", out), ("dout", dout), ("lse", lse)], what)
    _shape_check(q.dim() == 4 and k.dim() == 4, what, "q and k must be [N,S,H,D]")
    n, h, sq, sk, d = _attn_dims(q, k, v, bias, kmask, what, nshd=True)
    code = _dtype_code(q, (_native.F16, _native.BF16), what)
    _shape_check(out.shape == q.shape and out.dtype == q.dtype, what,
                 "out must match q")
    _shape_check(dout.shape == q.shape and dout.dtype == q.dtype, what,
                 "dout must match q")
    _shape_check(lse.shape == (n, h, sq) and lse.dtype == torch.float32, what,
                 "lse must be float32 [N,H,Sq]")
    if scale is None:
        scale = 1.0 / math.sqrt(d)
    lib = _native.lib()
    ws_bytes = lib.clk_attention_bwd_workspace_size(n, h, sq, sk, d)
    ws = _workspace(q, ws_bytes)
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    dbias = q.new_empty((h, sq, sk), dtype=torch.float32)
    _launch(index, lib.clk_attention_bwd_nshd, code, q.data_ptr(), k.data_ptr(), v.data_ptr(),
            bias.data_ptr(), _ptr(kmask), out.data_ptr(), dout.data_ptr(), lse.data_ptr(),
            dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), dbias.data_ptr(), ws.data_ptr(), ws_bytes,
            n, h, sq, sk, d, float(scale))
    return dq, dk, dv, dbias


def _ln_dims(x, scale, what):
    _shape_check(x.dim() >= 1, what, "x must have at least one axis")
    c = x.shape[-1]
    m = x.numel() // c if c else 0
    _shape_check(scale.shape == (c,) and scale.dtype == torch.float32, what,
                 "scale must be float32 [C]")
    return m, c


def layer_norm(x, scale, offset, eps=1e-5):
    """LayerNorm over the last axis of x (f16, bf16 or f32); scale and offset float32 [C]."""
    what = "layer_norm"
    index = _require([("x", x), ("scale", scale), ("offset", offset)], what)
    m, c = _ln_dims(x, scale, what)
    _shape_check(offset.shape == (c,) and offset.dtype == torch.float32, what,
                 "offset must be float32 [C]")
    code = _dtype_code(x, (_native.F16, _native.BF16, _native.F32), what)
    y = torch.empty_like(x)
    _launch(index, _native.lib().clk_layer_norm_fwd, code, x.data_ptr(), scale.data_ptr(),
            offset.data_ptr(), y.data_ptr(), m, c, float(eps))
    return y


def layer_norm_bwd(x, scale, dy, eps=1e-5):
    """(dx, dscale, doffset); dscale and doffset are float32 [C]."""
    what = "layer_norm_bwd"
    index = _require([("x", x), ("scale", scale), ("dy", dy)], what)
    m, c = _ln_dims(x, scale, what)
    _shape_check(dy.shape == x.shape and dy.dtype == x.dtype, what,
                 "dy must match x")
    code = _dtype_code(x, (_native.F16, _native.BF16, _native.F32), what)
    lib = _native.lib()
    ws_bytes = lib.clk_layer_norm_bwd_workspace_size(m, c)
    ws = _workspace(x, ws_bytes)
    dx = torch.empty_like(x)
    dscale = x.new_empty(c, dtype=torch.float32)
    doffset = x.new_empty(c, dtype=torch.float32)
    _launch(index, lib.clk_layer_norm_bwd, code, x.data_ptr(), scale.data_ptr(), dy.data_ptr(),
            dx.data_ptr(), dscale.data_ptr(), doffset.data_ptr(), ws.data_ptr(), ws_bytes, m, c,
            float(eps))
    return dx, dscale, doffset


def gated_dual_proj(x, wp, bp, wg, bg, mask):
    """mask[m] * (x.wp + bp) * sigmoid(x.wg + bg) for x [M,K], wp/wg [K,N], bp/bg [N], mask [M]."""
    what = "gated_dual_proj"
    index = _require([("x", x), ("wp", wp), ("bp", bp), ("wg", wg), ("bg", bg), ("mask", mask)],
                     what)
    _shape_check(x.dim() == 2, what, "x must be [M,K]")
    m, kdim = x.shape
    _shape_check(wp.dim() == 2 and wp.shape[0] == kdim, what, "wp must be [K,N]")
    n = wp.shape[1]
    _shape_check(wg.shape == (kdim, n), what, "wg must be [K,N]")
    _shape_check(bp.shape == (n,) and bg.shape == (n,), what, "bp, bg must be [N]")
    _shape_check(mask.shape == (m,), what, "mask must be [M]")
    _shape_check(_all_dtype(x.dtype, (wp, bp, wg, bg, mask)), what,
                 "all operands must share one dtype")
    code = _dtype_code(x, (_native.F16, _native.BF16), what)
    out = x.new_empty((m, n))
    _launch(index, _native.lib().clk_gated_dual_proj, code, x.data_ptr(), wp.data_ptr(),
            bp.data_ptr(), wg.data_ptr(), bg.data_ptr(), mask.data_ptr(), out.data_ptr(), m, kdim,
            n)
    return out


def gated_dual_proj_bwd(x, wp, bp, wg, bg, mask, dout, dx=None):
    """Gradients of gated_dual_proj: (dx, dwp, dbp, dwg, dbg); dx in x's dtype, the rest
    float32. If dx is given, the input gradient is added to it in place (two branches that read
    the same x)."""
    what = "gated_dual_proj_bwd"
    index = _require([("x", x), ("wp", wp), ("bp", bp), ("wg", wg), ("bg", bg), ("mask", mask),
                      ("dout", dout), ("dx", dx)], what)
    _shape_check(x.dim() == 2, what, "x must be [M,K]")
    m, kdim = x.shape
    _shape_check(wp.dim() == 2 and wp.shape[0] == kdim, what, "wp must be [K,N]")
    n = wp.shape[1]
    _shape_check(wg.shape == (kdim, n), what, "wg must be [K,N]")
    _shape_check(bp.shape == (n,) and bg.shape == (n,), what, "bp, bg must be [N]")
    _shape_check(mask.shape == (m,), what, "mask must be [M]")
    _shape_check(dout.shape == (m, n), what, "dout must be [M,N]")
    _shape_check(_all_dtype(x.dtype, (wp, bp, wg, bg, mask, dout)), what,
                 "all operands must share one dtype")
    code = _dtype_code(x, (_native.F16, _native.BF16), what)
    acc = dx is not None
    if acc:
        _shape_check(dx.shape == (m, kdim) and dx.dtype == x.dtype, what,
                     "dx must be [M,K] of x's dtype")
    else:
        dx = torch.empty_like(x)
    f32 = dict(dtype=torch.float32)
    dwp, dwg = x.new_empty((kdim, n), **f32), x.new_empty((kdim, n), **f32)
    dbp, dbg = x.new_empty(n, **f32), x.new_empty(n, **f32)
    lib = _native.lib()
    wsb = lib.clk_gated_dual_proj_bwd_workspace_size(m, kdim, n)
    ws = _workspace(x, wsb)
    _launch(index, lib.clk_gated_dual_proj_bwd, code, x.data_ptr(), wp.data_ptr(), bp.data_ptr(),
            wg.data_ptr(), bg.data_ptr(), mask.data_ptr(), dout.data_ptr(), dx.data_ptr(),
            dwp.data_ptr(), dbp.data_ptr(), dwg.data_ptr(), dbg.data_ptr(), ws.data_ptr(), wsb, m,
            kdim, n, 1 if acc else 0)
    return dx, dwp, dbp, dwg, dbg


def ln_gated_dual_proj_bwd(z, ln_scale, ln_offset, branch_a, branch_b, mask, da, db, eps=1e-5):
    """Gradients of ln_gated_dual_proj: (dz, dln_scale, dln_offset, grads_a, grads_b) with
    grads_x = (dwp, dbp, dwg, dbg). Recomputes y = LN(z), runs the GDP backward of both branches
    into one dy, then the LayerNorm backward."""
    y = layer_norm(z, ln_scale, ln_offset, eps)
    c = z.shape[-1]
    y2, m2 = y.reshape(-1, c), mask.reshape(-1)
    dy, *ga = gated_dual_proj_bwd(y2, *branch_a, m2, da.reshape(y2.shape[0], -1))
    _, *gb = gated_dual_proj_bwd(y2, *branch_b, m2, db.reshape(y2.shape[0], -1), dx=dy)
    dz, dsc, dof = layer_norm_bwd(z, ln_scale, dy.reshape(z.shape), eps)
    return dz, dsc, dof, tuple(ga), tuple(gb)


def ln_gated_dual_proj(z, ln_scale, ln_offset, branch_a, branch_b, mask, eps=1e-5):
    """(a, b): LayerNorm(z) then both gated projections, in one pass. Each branch is
    (wp, bp, wg, bg); z [M,C] (or [..., C]); mask [M]."""
    what = "ln_gated_dual_proj"
    wpa, bpa, wga, bga = branch_a
    wpb, bpb, wgb, bgb = branch_b
    index = _require([("z", z), ("ln_scale", ln_scale), ("ln_offset", ln_offset), ("wpa", wpa),
                      ("bpa", bpa), ("wga", wga), ("bga", bga), ("wpb", wpb), ("bpb", bpb),
                      ("wgb", wgb), ("bgb", bgb), ("mask", mask)], what)
    m, c = _ln_dims(z, ln_scale, what)
    _shape_check(wpa.dim() == 2 and wpa.shape[0] == c, what, "weights must be [C,N]")
    n = wpa.shape[1]
    for name, w in (("wga", wga), ("wpb", wpb), ("wgb", wgb)):
        if w.shape != (c, n):
            _fail(what, "%s must be [C,N]" % name)
    for name, b in (("bpa", bpa), ("bga", bga), ("bpb", bpb), ("bgb", bgb)):
        if b.shape != (n,):
            _fail(what, "%s must be [N]" % name)
    _shape_check(mask.numel() == m, what, "mask must have M elements")
    code = _dtype_code(z, (_native.F16, _native.BF16), what)
    a = z.new_empty(tuple(z.shape[:-1]) + (n,))
    b = torch.empty_like(a)
    _launch(index, _native.lib().clk_ln_gated_dual_proj, code, z.data_ptr(), ln_scale.data_ptr(),
            ln_offset.data_ptr(), wpa.data_ptr(), bpa.data_ptr(), wga.data_ptr(), bga.data_ptr(),
            wpb.data_ptr(), bpb.data_ptr(), wgb.data_ptr(), bgb.data_ptr(), mask.data_ptr(),
            a.data_ptr(), b.data_ptr(), m, c, n, float(eps))
    return a, b


def ln_pair_bias(z, scale, offset, w, eps=1e-5):
    """LN(z).w transposed to the attention bias layout: z [Sq,Sk,C] (or [M,C]), scale/offset
    float32 [C], w [C,H] -> [H,Sq,Sk] (or [H,M])."""
    what = "ln_pair_bias"
    index = _require([("z", z), ("scale", scale), ("offset", offset), ("w", w)], what)
    m, c = _ln_dims(z, scale, what)
    _shape_check(w.dim() == 2 and w.shape[0] == c and w.dtype == z.dtype, what,
                 "w must be [C,H] of z's dtype")
    _shape_check(offset.shape == (c,) and offset.dtype == torch.float32, what,
                 "offset must be float32 [C]")
    h = w.shape[1]
    code = _dtype_code(z, (_native.F16, _native.BF16), what)
    out = z.new_empty((h,) + tuple(z.shape[:-1]))
    _launch(index, _native.lib().clk_ln_pair_bias, code, z.data_ptr(), scale.data_ptr(),
            offset.data_ptr(), w.data_ptr(), out.data_ptr(), m, c, h, float(eps))
    return out


def attention_gate(o, x, wg, bg):
    """o * sigmoid(x.wg + bg), transposed to the output projection's layout: o [N,H,Sq,D] (the
    attention output), x [N,Sq,C], wg [C,H*D], bg [H*D] -> [N,Sq,H*D]."""
    what = "attention_gate"
    index = _require([("o", o), ("x", x), ("wg", wg), ("bg", bg)], what)
    _shape_check(o.dim() == 4, what, "o must be [N,H,Sq,D]")
    n, h, sq, d = o.shape
    _shape_check(x.dim() == 3 and tuple(x.shape[:2]) == (n, sq), what, "x must be [N,Sq,C]")
    c = x.shape[2]
    _shape_check(wg.shape == (c, h * d), what, "wg must be [C,H*D]")
    _shape_check(bg.shape == (h * d,), what, "bg must be [H*D]")
    _shape_check(_all_dtype(o.dtype, (x, wg, bg)), what,
                 "all operands must share one dtype")
    code = _dtype_code(o, (_native.F16, _native.BF16), what)
    out = o.new_empty((n, sq, h * d))
    _launch(index, _native.lib().clk_attention_gate, code, o.data_ptr(), x.data_ptr(),
            wg.data_ptr(), bg.data_ptr(), out.data_ptr(), n, h, sq, d, c)
    return out


def attention_gate_bwd(o, x, wg, bg, dout, dx=None):
    """Gradients of attention_gate for dout [N,Sq,H*D]: (do, dx, dwg, dbg) with do [N,H,Sq,D]
    (the dout of attention_bwd) and dx [N,Sq,C] in o's dtype, dwg [C,H*D] and dbg [H*D] float32.
    If dx is given, the input gradient is added to it in place (x also feeds the q, k, v
    projections)."""
    what = "attention_gate_bwd"
    index = _require([("o", o), ("x", x), ("wg", wg), ("bg", bg), ("dout", dout), ("dx", dx)],
                     what)
    _shape_check(o.dim() == 4, what, "o must be [N,H,Sq,D]")
    n, h, sq, d = o.shape
    _shape_check(x.dim() == 3 and tuple(x.shape[:2]) == (n, sq), what, "x must be [N,Sq,C]")
    c = x.shape[2]
    _shape_check(wg.shape == (c, h * d), what, "wg must be [C,H*D]")
    _shape_check(bg.shape == (h * d,), what, "bg must be [H*D]")
    _shape_check(dout.shape == (n, sq, h * d), what, "dout must be [N,Sq,H*D]")
    _shape_check(_all_dtype(o.dtype, (x, wg, bg, dout)), what,
                 "all operands must share one dtype")
    code = _dtype_code(o, (_native.F16, _native.BF16), what)
    acc = dx is not None
    if acc:
        _shape_check(dx.shape == (n, sq, c) and dx.dtype == o.dtype, what,
                     "dx must be [N,Sq,C] of o's dtype")
    else:
        dx = torch.empty_like(x)
    do = torch.empty_like(o)
    f32 = dict(dtype=torch.float32)
    dwg, dbg = o.new_empty((c, h * d), **f32), o.new_empty(h * d, **f32)
    lib = _native.lib()
    wsb = lib.clk_attention_gate_bwd_workspace_size(n, h, sq, d, c)
    ws = _workspace(o, wsb)
    _launch(index, lib.clk_attention_gate_bwd, code, o.data_ptr(), x.data_ptr(), wg.data_ptr(),
            bg.data_ptr(), dout.data_ptr(), do.data_ptr(), dx.data_ptr(), dwg.data_ptr(),
            dbg.data_ptr(), ws.data_ptr(), wsb, n, h, sq, d, c, 1 if acc else 0)
    return do, dx, dwg, dbg


def _gated_call(q, k, v, bias, kmask, x, wg, bg, scale, residuals, what):
    index = _require([("q", q), ("k", k), ("v", v), ("bias", bias), ("kmask", kmask), ("x", x),
                      ("wg", wg), ("bg", bg)], what)
    n, h, sq, sk, d = _attn_dims(q, k, v, bias, kmask, what)
    _shape_check(x.dim() == 3 and tuple(x.shape[:2]) == (n, sq), what, "x must be [N,Sq,C]")
    c = x.shape[2]
    _shape_check(wg.shape == (c, h * d), what, "wg must be [C,H*D]")
    _shape_check(bg.shape == (h * d,), what, "bg must be [H*D]")
    _shape_check(_all_dtype(q.dtype, (x, wg, bg)), what,
                 "x, wg and bg must have the dtype of q")
    code = _dtype_code(q, (_native.F16, _native.BF16), what)
    if scale is None:
        scale = 1.0 / math.sqrt(d)
    gated = q.new_empty((n, sq, h * d))
    out = torch.empty_like(q) if residuals else None
    lse = q.new_empty((n, h, sq), dtype=torch.float32) if residuals else None
    _launch(index, _native.lib().clk_attention_fwd_gated, code, q.data_ptr(), k.data_ptr(),
            v.data_ptr(), bias.data_ptr(), _ptr(kmask), x.data_ptr(), wg.data_ptr(), bg.data_ptr(),
            gated.data_ptr(), _ptr(out), _ptr(lse), n, h, sq, sk, d, c, float(scale))
    return gated, out, lse


def attention_gated(q, k, v, bias, kmask, x, wg, bg, scale=None):
    """attention(q, k, v, bias, kmask) gated by sigmoid(x.wg + bg) in one kernel, in the output
    projection's layout: q [N,H,Sq,D], k/v [N,H,Sk,D], bias [H,Sq,Sk], kmask uint8 [N,Sk] or
    None, x [N,Sq,C] with C % 32 == 0, wg [C,H*D], bg [H*D] -> [N,Sq,H*D]. The ungated
    attention output never reaches memory."""
    gated, _, _ = _gated_call(q, k, v, bias, kmask, x, wg, bg, scale, False, "attention_gated")
    return gated


def attention_gated_fwd(q, k, v, bias, kmask, x, wg, bg, scale=None):
    """(gated, out, lse): attention_gated plus the ungated output [N,H,Sq,D] and the float32
    logsumexp [N,H,Sq] that attention_bwd needs."""
    return _gated_call(q, k, v, bias, kmask, x, wg, bg, scale, True, "attention_gated_fwd")


def triangle_einsum(a, b):
    """x[c] = a[c] . b[c]^T for channel-major a, b [C,N,N] (the triangle-multiplication
    contraction with the channel index first and the contracted index last); N % 8 == 0."""
    what = "triangle_einsum"
    index = _require([("a", a), ("b", b)], what)
    _shape_check(a.dim() == 3 and a.shape[1] == a.shape[2], what, "a must be [C,N,N]")
    _shape_check(b.shape == a.shape and b.dtype == a.dtype, what,
                 "b must match a")
    c, n, _ = a.shape
    code = _dtype_code(a, (_native.F16, _native.BF16), what)
    x = torch.empty_like(a)
    _launch(index, _native.lib().clk_triangle_einsum, code, a.data_ptr(), b.data_ptr(),
            x.data_ptr(), c, n)
    return x


def triangle_multiply(z, mask, ln_in, weights, biases, ln_center, outgoing=True, eps=1e-5):
    """AlphaFold's triangle multiplication on the pair representation z [N,N,C] with mask [N,N].
    ln_in, ln_center: (scale, offset) float32 [C]; weights: the six [C,C] matrices (left
    projection, right projection, left gate, right gate, output projection, output gate), biases
    their [C] vectors, all of z's dtype. Returns [N,N,C]."""
    what = "triangle_multiply"
    ws6, bs6 = list(weights), list(biases)
    _shape_check(len(ws6) == 6 and len(bs6) == 6, what, "six weights and six biases")
    lns = [ln_in[0], ln_in[1], ln_center[0], ln_center[1]]
    index = _require([("z", z), ("mask", mask)] + [("w%d" % i, w) for i, w in enumerate(ws6)]
                     + [("b%d" % i, b) for i, b in enumerate(bs6)]
                     + [("ln%d" % i, t) for i, t in enumerate(lns)], what)
    _shape_check(z.dim() == 3 and z.shape[0] == z.shape[1], what, "z must be [N,N,C]")
    n, _, c = z.shape
    _shape_check(mask.shape == (n, n) and mask.dtype == z.dtype, what,
                 "mask must be [N,N] of z's dtype")
    _shape_check(all(w.shape == (c, c) and w.dtype == z.dtype for w in ws6), what,
                 "weights must be [C,C] of z's dtype")
    _shape_check(all(b.shape == (c,) and b.dtype == z.dtype for b in bs6), what,
                 "biases must be [C] of z's dtype")
    _shape_check(all(t.shape == (c,) and t.dtype == torch.float32 for t in lns), what,
                 "LayerNorm scales and offsets must be float32 [C]")
    code = _dtype_code(z, (_native.F16, _native.BF16), what)
    lib = _native.lib()
    wsb = lib.clk_triangle_multiply_workspace_size(n, c)
    ws = _workspace(z, wsb)
    out = torch.empty_like(z)
    arr = lambda ts: (ctypes.c_void_p * len(ts))(*[t.data_ptr() for t in ts])  # noqa: E731
    _launch(index, lib.clk_triangle_multiply, code, z.data_ptr(), mask.data_ptr(), arr(lns),
            arr(ws6), arr(bs6), out.data_ptr(), ws.data_ptr(), wsb, n, c, 1 if outgoing else 0,
            float(eps))
    return out


class AttentionFunction(torch.autograd.Function):
    """Differentiable attention: forward saves (out, lse); backward calls attention_bwd."""

    @staticmethod
    def forward(ctx, q, k, v, bias, kmask, scale):
        out, lse = attention_fwd(q, k, v, bias, kmask, scale)
        ctx.save_for_backward(q, k, v, bias, kmask, out, lse)
        ctx.scale = scale
        return out

    @staticmethod
    def backward(ctx, dout):
        q, k, v, bias, kmask, out, lse = ctx.saved_tensors
        dq, dk, dv, dbias = attention_bwd(q, k, v, bias, kmask, out, dout.contiguous(), lse,
                                          ctx.scale)
        return dq, dk, dv, dbias.to(bias.dtype), None, None


class GatedAttentionFunction(torch.autograd.Function):
    """Differentiable gated attention, o(q, k, v, bias, kmask) * sigmoid(x.wg + bg) in the output
    projection's [N,Sq,H*D] layout. forward: attention_gated_fwd (one launch) when fused, else
    attention_fwd then attention_gate (the faster pair on MSA row shapes); both keep the ungated
    output and the logsumexp. backward: attention_gate_bwd (do, dx, dwg, dbg), then
    attention_bwd with that do. Gradients for q, k, v, bias, x, wg, bg."""

    @staticmethod
    def forward(ctx, q, k, v, bias, kmask, x, wg, bg, scale, fused=False):
        if fused:
            gated, out, lse = attention_gated_fwd(q, k, v, bias, kmask, x, wg, bg, scale)
        else:
            out, lse = attention_fwd(q, k, v, bias, kmask, scale)
            gated = attention_gate(out, x, wg, bg)
        ctx.save_for_backward(q, k, v, bias, kmask, x, wg, bg, out, lse)
        ctx.scale = scale
        return gated

    @staticmethod
    def backward(ctx, dgated):
        q, k, v, bias, kmask, x, wg, bg, out, lse = ctx.saved_tensors
        do, dx, dwg, dbg = attention_gate_bwd(out, x, wg, bg, dgated.contiguous())
        dq, dk, dv, dbias = attention_bwd(q, k, v, bias, kmask, out, do, lse, ctx.scale)
        return (dq, dk, dv, dbias.to(bias.dtype), None, dx, dwg.to(wg.dtype), dbg.to(bg.dtype),
                None, None)


class LayerNormFunction(torch.autograd.Function):
    """Differentiable LayerNorm over the last axis (statistics recomputed in backward)."""

    @staticmethod
    def forward(ctx, x, scale, offset, eps):
        ctx.save_for_backward(x, scale)
        ctx.eps = eps
        return layer_norm(x, scale, offset, eps)

    @staticmethod
    def backward(ctx, dy):
        x, scale = ctx.saved_tensors
        dx, dscale, doffset = layer_norm_bwd(x, scale, dy.contiguous(), ctx.eps)
        return dx, dscale, doffset, None
