"""Attention forward on the GPU against the float64 oracle (through the C ABI)."""
import numpy as np
import pytest
import torch

from _util import TOL, assert_close, dname, np64
from colabfold_legacy_kernels import _native, ops
from colabfold_legacy_kernels.workloads import attention_inputs, attention_workload, gate_inputs
from oracle import attention as ref
from oracle import gate as ref_gate

pytestmark = pytest.mark.gpu

# (N, H, Sq, Sk, D, masked_tail, masked_rows): aligned, ragged, every head dim, masks.
CASES = [
    (2, 2, 64, 64, 32, 0.0, 0),
    (3, 2, 100, 77, 32, 0.1, 1),
    (2, 1, 130, 200, 64, 0.2, 0),
    (2, 4, 64, 64, 16, 0.0, 1),
    (2, 2, 48, 40, 8, 0.1, 0),
    (1, 1, 1, 1, 32, 0.0, 0),
    (2, 3, 257, 129, 32, 0.05, 1),
    (2, 2, 33, 300, 64, 0.0, 0),
    (1, 1, 16, 4100, 32, 0.1, 0),  # more than 64 key tiles, ragged last tile
    (1, 1, 16, 16400, 32, 0.1, 0),  # more key tiles than the masked-bias patching covers
    (3, 2, 64, 320, 32, 0.6, 1),    # a padding tail of whole key tiles
    # Biases over 2 MB run the head-outer work-item order in groups of rows: 13 rows in groups
    # of 9 and 4 (a ragged last group), and 5 rows in one group smaller than the group size.
    (13, 4, 640, 640, 32, 0.1, 1),
    (5, 2, 1024, 1024, 16, 0.0, 0),
]


def _oracle(inp, rows=None):
    sel = slice(None) if rows is None else rows
    return ref.attention_fwd(np64(inp["q"][sel]), np64(inp["k"][sel]), np64(inp["v"][sel]),
                             np64(inp["bias"]), inp["kmask"][sel].cpu().numpy(), inp["scale"])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=dname)
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:5])))
def test_attention_fwd_parity(cuda, case, dtype):
    n, h, sq, sk, d, tail, rows = case
    inp = attention_inputs(n, h, sq, sk, d, dtype, seed=sq * 7 + sk, bias_var=1.0,
                           masked_tail=tail, masked_rows=rows, with_dout=False)
    g = {k: (v.to(cuda) if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    out, lse = ops.attention_fwd(g["q"], g["k"], g["v"], g["bias"], g["kmask"], g["scale"])
    o_ref, lse_ref = _oracle(inp)
    tol = TOL[dname(dtype)]["o"]
    assert_close("O", out, o_ref, tol)
    # lse is float32 from float32 logits: absolute error on the logit scale. A row with no
    # present key reports ln(Sk) (relative to its masked logit); the oracle's value is
    # -1e9 + ln(Sk), which float32 cannot hold.
    empty = (inp["kmask"].numpy() == 0).all(axis=1)[:, None, None]
    lse_ref = np.where(empty, np.log(sk), lse_ref)
    assert np.abs(np64(lse) - lse_ref).max() < 5e-2
    # The inference entry (VoltaMma contract) gives the same bits as the training entry.
    out2 = ops.attention(g["q"], g["k"], g["v"], g["bias"], g["kmask"], g["scale"], 64, 64)
    assert torch.equal(out, out2)


# (N, H, Sq, Sk, D, masked_tail, masked_rows): every head dim, one- and two-sub-tile query
# blocks, the bias-tile and element-wise paths (Sk % 8), a padding tail, rows with no key, H = 1.
NSHD_CASES = [(3, 4, 100, 77, 32, 0.1, 1), (2, 2, 64, 384, 32, 0.2, 1),
              (2, 3, 130, 200, 64, 0.0, 0), (2, 4, 48, 40, 8, 0.1, 0), (2, 2, 33, 136, 16, 0.0, 1),
              (4, 1, 70, 96, 32, 0.5, 0)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=dname)
@pytest.mark.parametrize("case", NSHD_CASES, ids=lambda c: "x".join(map(str, c[:5])))
def test_attention_fwd_nshd_layout(cuda, case, dtype):
    """The [N,S,H,D] entry runs the same kernel with rows H*D apart: O (in [N,S,H,D]) and lse
    are bit-identical to the [N,H,S,D] entry on the transposed operands, and match the oracle."""
    n, h, sq, sk, d, tail, rows = case
    inp = attention_inputs(n, h, sq, sk, d, dtype, seed=sq * 5 + sk + d, bias_var=1.0,
                           masked_tail=tail, masked_rows=rows, with_dout=False)
    g = {k: (v.to(cuda) if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    out, lse = ops.attention_fwd(g["q"], g["k"], g["v"], g["bias"], g["kmask"], g["scale"])
    t = lambda x: x.transpose(1, 2).contiguous()  # [N,H,S,D] <-> [N,S,H,D]
    out_s, lse_s = ops.attention_nshd(t(g["q"]), t(g["k"]), t(g["v"]), g["bias"], g["kmask"],
                                      g["scale"], want_lse=True)
    assert out_s.shape == (n, sq, h, d)
    assert torch.equal(t(out_s), out)
    assert torch.equal(lse_s, lse)
    assert_close("O", t(out_s), _oracle(inp)[0], TOL[dname(dtype)]["o"])
    out_n, lse_n = ops.attention_nshd(t(g["q"]), t(g["k"]), t(g["v"]), g["bias"], g["kmask"],
                                      g["scale"])
    assert lse_n is None and torch.equal(out_n, out_s)


# (N, H, Sq, Sk, D): whole and ragged key tiles, the element-wise mask path (Sk % 8 != 0).
MIXED_MASK_SHAPES = [(8, 2, 70, 200, 32), (6, 2, 64, 77, 32), (6, 2, 40, 456, 16),
                     (4, 1, 130, 384, 64), (5, 2, 64, 136, 8)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=dname)
@pytest.mark.parametrize("shape", MIXED_MASK_SHAPES, ids=lambda c: "x".join(map(str, c)))
def test_attention_fwd_mixed_masks(cuda, shape, dtype):
    """Per-row masks of every kind in one call: random holes with a padding tail, a row with no
    present key, a row whose first 64-key tile is entirely absent (its running max starts on
    absent keys), a row with everything present, and one whose only present key is the last."""
    n, h, sq, sk, d = shape
    inp = attention_inputs(n, h, sq, sk, d, dtype, seed=sk + 3 * n, with_dout=False)
    gen = torch.Generator().manual_seed(sk * 5 + n)
    km = (torch.rand((n, sk), generator=gen) > 0.2).to(torch.uint8)
    km[:, sk - sk // 5:] = 0
    km[1] = 0
    km[2, :min(64, sk - 1)] = 0
    km[2, sk - 1] = 1
    km[3] = 1
    km[n - 1] = 0
    km[n - 1, sk - 1] = 1
    inp["kmask"] = km
    g = {k: (v.to(cuda) if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    out, lse = ops.attention_fwd(g["q"], g["k"], g["v"], g["bias"], g["kmask"], g["scale"])
    o_ref, lse_ref = _oracle(inp)
    assert_close("O", out, o_ref, TOL[dname(dtype)]["o"])
    empty = (km.numpy() == 0).all(axis=1)[:, None, None]
    lse_ref = np.where(empty, np.log(sk), lse_ref)
    assert np.abs(np64(lse) - lse_ref).max() < 5e-2


def test_attention_fwd_no_mask_is_all_present(cuda):
    inp = attention_inputs(2, 2, 64, 96, 32, torch.bfloat16, seed=5, with_dout=False)
    g = {k: (v.to(cuda) if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    a = ops.attention(g["q"], g["k"], g["v"], g["bias"], None, g["scale"])
    b = ops.attention(g["q"], g["k"], g["v"], g["bias"], torch.ones_like(g["kmask"]), g["scale"])
    assert torch.equal(a, b)


def test_attention_fwd_fully_masked_row_is_mean_v(cuda):
    """jnp's float32 additive mask: a row with every key masked attends uniformly over its Sk
    keys (not over tile padding), so O = mean(V)."""
    inp = attention_inputs(2, 2, 40, 70, 32, torch.bfloat16, seed=9, with_dout=False)
    inp["kmask"][1] = 0
    g = {k: (v.to(cuda) if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    out = ops.attention(g["q"], g["k"], g["v"], g["bias"], g["kmask"], g["scale"])
    mean_v = np64(inp["v"][1]).mean(axis=1, keepdims=True).repeat(40, axis=1)
    assert_close("O[masked]", out[1], mean_v, TOL["bf16"]["o"])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=dname)
@pytest.mark.parametrize("slope", [0.02, 0.06, 0.3, -0.3])
def test_attention_fwd_rising_and_falling_logits(cuda, slope, dtype):
    """Bias ramps along the keys, so a row's running max rises tile after tile by less than,
    about, or more than the forward's rescale slack (2^8 in P: 5.5 logit units; a 64-key tile
    rises by 64*slope), or falls (slope < 0: the first tile holds the max). O and the
    logsumexp against the oracle."""
    n, h, sq, sk, d = 2, 2, 70, 320, 32
    inp = attention_inputs(n, h, sq, sk, d, dtype, seed=13, bias_var=0.25, masked_tail=0.05,
                           with_dout=False)
    ramp = slope * torch.arange(sk, dtype=torch.float32)
    inp["bias"] = (inp["bias"].float() + ramp).to(dtype)
    g = {k: (v.to(cuda) if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    out, lse = ops.attention_fwd(g["q"], g["k"], g["v"], g["bias"], g["kmask"], g["scale"])
    o_ref, lse_ref = _oracle(inp)
    assert_close("O", out, o_ref, TOL[dname(dtype)]["o"])
    assert np.abs(np64(lse) - lse_ref).max() < 5e-2


# Every (D, block_q, block_k) that VoltaMma (cuda/volta_mma_attn.cu:323-331) or VoltaWmma
# (cuda/volta_wmma_attn.cu:286-292) dispatches, plus one neither knows: block sizes are hints.
REFERENCE_BLOCKS = {
    8: [(64, 64), (64, 32), (32, 32), (128, 64), (32, 64), (7, 5)],
    16: [(64, 64), (32, 32), (64, 32)],
    32: [(64, 64), (64, 32), (32, 64), (32, 32), (128, 64), (16, 64), (128, 32), (7, 5)],
    64: [(64, 64), (32, 32), (64, 32)],
}


@pytest.mark.parametrize("d,block", [(d, b) for d, bs in REFERENCE_BLOCKS.items() for b in bs],
                         ids=lambda v: str(v))
def test_attention_fwd_accepts_reference_block_hints(cuda, d, block):
    inp = attention_inputs(1, 2, 70, 90, d, torch.float16, seed=3, masked_tail=0.1,
                           with_dout=False)
    g = {k: (v.to(cuda) if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    base = ops.attention(g["q"], g["k"], g["v"], g["bias"], g["kmask"], g["scale"])
    out = ops.attention(g["q"], g["k"], g["v"], g["bias"], g["kmask"], g["scale"], *block)
    assert torch.equal(base, out)
    o_ref, _ = _oracle(inp)
    assert_close("O", out, o_ref, TOL["f16"]["o"])


@pytest.mark.parametrize("name", ["triangle_attn_256", "triangle_attn_384", "msa_row_attn",
                                  "triangle_attn_1024"])
def test_attention_fwd_full_size_rows(cuda, name):
    """Full workload on the GPU; sampled rows n against the oracle (rows are independent),
    including two fully padded rows (no present key) where the workload has them."""
    inp = attention_workload(name, torch.bfloat16, device=cuda, with_dout=False)
    out, lse = ops.attention_fwd(inp["q"], inp["k"], inp["v"], inp["bias"], inp["kmask"],
                                 inp["scale"])
    n = inp["q"].shape[0]
    padded = (inp["kmask"] == 0).all(dim=1).nonzero().flatten().tolist()
    if name == "msa_row_attn":
        assert len(padded) == 102
    rows = sorted({0, 1, n // 2, n - 1} | set(padded[:1] + padded[-1:]))
    cpu = {k: (v.cpu() if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    o_ref, _ = _oracle(cpu, rows)
    assert_close("O[rows]", out[rows], o_ref, TOL["bf16"]["o"])
    assert torch.isfinite(lse).all()


def test_attention_rejects_bad_operands(cuda):
    inp = attention_inputs(1, 2, 16, 16, 32, torch.bfloat16, seed=1, with_dout=False)
    g = {k: (v.to(cuda) if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    with pytest.raises(ops.InvalidArgument):
        ops.attention(g["q"], g["k"], g["v"], g["bias"][:, :8], g["kmask"])
    q24 = torch.zeros((1, 2, 16, 24), device=cuda, dtype=torch.bfloat16)
    with pytest.raises(ops.InvalidArgument):
        ops.attention(q24, q24, q24, g["bias"], g["kmask"])
    with pytest.raises(ops.InvalidArgument):
        ops.attention(g["q"], g["k"], g["v"], g["bias"], g["kmask"], None, 0, 64)


@pytest.mark.parametrize("gated", [False, True], ids=["plain", "gated"])
def test_attention_fwd_nan_propagates(cuda, gated):
    """A NaN in one query row, and a NaN bias entry at one present key, make exactly the output
    rows they reach NaN (every head dim), with and without the fused gate; every other row stays
    finite. (The forward's device code assumes no NaN operand for its maxima; the exponentials
    and the sums still carry a NaN score into its row.)"""
    n, h, sq, sk, d = 2, 4, 70, 96, 32
    inp = attention_inputs(n, h, sq, sk, d, torch.bfloat16, seed=5, masked_tail=0.1,
                           with_dout=False)
    q, bias = inp["q"].clone(), inp["bias"].clone()
    q[1, 2, 5, 3] = float("nan")
    bias[3, 40, 17] = float("nan")  # key 17 is present in every row
    g = {k: (v.to(cuda) if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    g["q"], g["bias"] = q.to(cuda), bias.to(cuda)
    nan_rows = torch.zeros((n, h, sq), dtype=torch.bool)
    nan_rows[1, 2, 5] = True
    nan_rows[:, 3, 40] = True
    if gated:
        c = 128
        x, wg, bg = gate_inputs(n, sq, c, h * d, torch.bfloat16, seed=5, bias_std=0.5)
        out = ops.attention_gated(g["q"], g["k"], g["v"], g["bias"], g["kmask"], x.to(cuda),
                                  wg.to(cuda), bg.to(cuda), g["scale"]).cpu()
        out = out.reshape(n, sq, h, d).transpose(1, 2)
    else:
        out = ops.attention(g["q"], g["k"], g["v"], g["bias"], g["kmask"], g["scale"]).cpu()
    isnan = torch.isnan(out.float())
    assert isnan[nan_rows].all()
    assert torch.isfinite(out.float()[~nan_rows]).all()


def test_attention_row_with_no_weight(cuda):
    """Present-key logits below -5e8 (a bias of -1e9, the masked-logit convention, on every
    present key of one query row): that row has no weight, O = 0 and lse = +inf, and its
    gradients are zero; every other row is unaffected. The backward is compared with the oracle
    on inputs whose dO of that row is zero (which removes the row from every gradient there)."""
    n, h, sq, sk, d = 3, 2, 70, 96, 32
    inp = attention_inputs(n, h, sq, sk, d, torch.bfloat16, seed=8, masked_tail=0.1)
    b = inp["bias"].float()
    b[1, 20, :] = -1e9
    inp["bias"] = b.to(torch.bfloat16)
    inp["dout"][:, 1, 20, :] = 0
    g = {k: (v.to(cuda) if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    out, lse = ops.attention_fwd(g["q"], g["k"], g["v"], g["bias"], g["kmask"], g["scale"])
    assert torch.count_nonzero(out[:, 1, 20]).item() == 0
    assert torch.isinf(lse[:, 1, 20]).all() and (lse[:, 1, 20] > 0).all()
    o_ref, _ = _oracle(inp)
    assert_close("O[h0]", out[:, 0], o_ref[:, 0], TOL["bf16"]["o"])
    assert_close("O[h1, :20]", out[:, 1, :20], o_ref[:, 1, :20], TOL["bf16"]["o"])
    assert_close("O[h1, 21:]", out[:, 1, 21:], o_ref[:, 1, 21:], TOL["bf16"]["o"])
    dq, dk, dv, dbias = ops.attention_bwd(g["q"], g["k"], g["v"], g["bias"], g["kmask"], out,
                                          g["dout"], lse, g["scale"])
    assert torch.count_nonzero(dq[:, 1, 20]).item() == 0
    assert torch.count_nonzero(dbias[1, 20]).item() == 0
    rq, rk, rv, rb = ref.attention_bwd(np64(inp["q"]), np64(inp["k"]), np64(inp["v"]),
                                       np64(inp["bias"]), inp["kmask"].numpy(), inp["scale"],
                                       np64(inp["dout"]))
    tol = TOL["bf16"]["grad"]
    assert_close("dQ", dq, rq, tol)
    assert_close("dK", dk, rk, tol)
    assert_close("dV", dv, rv, tol)
    assert_close("dBias", dbias, rb, tol)


# (N, H, Sq, Sk, D): odd key counts around the edges of the 64-key tiles (blocks of one query
# parity, half of them with tiles that start at key -1), odd and even query counts around the
# edges of the 64- and 128-query blocks, one head (its odd biases read element by element) and
# even key counts that are no multiple of 8.
RAGGED_SHAPES = [(5, 2, 1, 1, 32), (5, 2, 2, 3, 8), (5, 4, 63, 63, 32), (5, 2, 64, 65, 16),
                 (5, 2, 65, 127, 32), (5, 3, 128, 129, 32), (5, 3, 129, 129, 32),
                 (5, 2, 255, 191, 8), (5, 2, 257, 193, 64), (5, 1, 130, 67, 32), (5, 2, 70, 66, 32),
                 (5, 3, 131, 190, 16), (5, 4, 515, 513, 32)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=dname)
@pytest.mark.parametrize("shape", RAGGED_SHAPES, ids=lambda c: "x".join(map(str, c)))
def test_attention_fwd_ragged_keys(cuda, shape, dtype):
    """Key counts that are no multiple of 8, with per-row masks: all present, none present, key 0
    absent, only the last key present, random holes. Both layouts, against the oracle."""
    n, h, sq, sk, d = shape
    inp = attention_inputs(n, h, sq, sk, d, dtype, seed=sk + 7 * sq, with_dout=False)
    gen = torch.Generator().manual_seed(sk + sq)
    km = torch.ones((n, sk), dtype=torch.uint8)
    km[1] = 0
    km[2, 0] = 0
    km[2, sk - 1] = 1
    km[3, :sk - 1] = 0
    km[4] = (torch.rand(sk, generator=gen) > 0.3).to(torch.uint8)
    km[4, sk // 2] = 1
    inp["kmask"] = km
    g = {k: (v.to(cuda) if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    out, lse = ops.attention_fwd(g["q"], g["k"], g["v"], g["bias"], g["kmask"], g["scale"])
    o_ref, lse_ref = _oracle(inp)
    assert_close("O", out, o_ref, TOL[dname(dtype)]["o"])
    empty = (km.numpy() == 0).all(axis=1)[:, None, None]
    assert np.abs(np64(lse) - np.where(empty, np.log(sk), lse_ref)).max() < 5e-2
    t = lambda x: x.transpose(1, 2).contiguous()  # noqa: E731
    out_s, lse_s = ops.attention_nshd(t(g["q"]), t(g["k"]), t(g["v"]), g["bias"], g["kmask"],
                                      g["scale"], want_lse=True)
    assert torch.equal(t(out_s), out) and torch.equal(lse_s, lse)
    # No mask and a mask of ones: the same bits, in both layouts.
    ones = torch.ones_like(g["kmask"])
    for scale in (g["scale"], -g["scale"]):
        args = (g["q"], g["k"], g["v"], g["bias"])
        out_1, lse_1 = ops.attention_fwd(*args, ones, scale)
        out_0, lse_0 = ops.attention_fwd(*args, None, scale)
        assert torch.equal(out_0, out_1) and torch.equal(lse_0, lse_1)
        out_t = ops.attention_nshd(*(t(x) for x in args[:3]), g["bias"], None, scale)[0]
        assert torch.equal(t(out_t), out_0)
        o_1, lse_r = _oracle({**inp, "kmask": torch.ones_like(km), "scale": scale})
        assert_close("O (no mask)", out_0, o_1, TOL[dname(dtype)]["o"])
        assert np.abs(np64(lse_0) - lse_r).max() < 5e-2
    # A negative scale takes the form without the bias MFMA at any key count.
    neg = {**inp, "scale": -inp["scale"]}
    out_n = ops.attention(g["q"], g["k"], g["v"], g["bias"], g["kmask"], neg["scale"])
    assert_close("O (negative scale)", out_n, _oracle(neg)[0], TOL[dname(dtype)]["o"])


# (Sq, Sk, D): one and two 64-query tiles past a block, odd and even numbers of tiles (odd ones
# round up to two per block in the larger blocks), both key parities, every head dim.
BLOCK_SHAPES = [(65, 66, 32), (128, 128, 16), (127, 129, 32), (130, 70, 64), (250, 96, 8),
                (193, 192, 32), (257, 64, 64), (300, 300, 16), (300, 65, 8), (513, 64, 32)]


@pytest.mark.parametrize("shape", BLOCK_SHAPES, ids=lambda c: "x".join(map(str, c)))
def test_attention_fwd_query_block_choice(cuda, shape):
    """Few rows run 64-query blocks, many rows the size that suits the shape: the same bits for
    every row either way, in both layouts and gated; the few rows against the oracle."""
    sq, sk, d = shape
    n, h = 5, 2
    inp = attention_inputs(n, h, sq, sk, d, torch.bfloat16, seed=sq + sk, masked_tail=0.2,
                           masked_rows=1, with_dout=False)
    x, wg, bg = (t.to(cuda) for t in gate_inputs(n, sq, 64, h * d, torch.bfloat16, seed=sk))
    g = {k: (v.to(cuda) if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    out, lse = ops.attention_fwd(g["q"], g["k"], g["v"], g["bias"], g["kmask"], g["scale"])
    assert_close("O", out, _oracle(inp)[0], TOL["bf16"]["o"])
    gated = ops.attention_gated(g["q"], g["k"], g["v"], g["bias"], g["kmask"], x, wg, bg,
                                g["scale"])
    reps = 1100 // (n * h * ((sq + 63) // 64)) + 1
    many = [t.repeat(reps, *[1] * (t.dim() - 1)) for t in (g["q"], g["k"], g["v"], g["kmask"], x)]
    q, k, v, km, xm = many
    t = lambda a: a.transpose(1, 2).contiguous()  # noqa: E731
    out_m, lse_m = ops.attention_fwd(q, k, v, g["bias"], km, g["scale"])
    out_s = ops.attention_nshd(t(q), t(k), t(v), g["bias"], km, g["scale"])[0]
    gated_m = ops.attention_gated(q, k, v, g["bias"], km, xm, wg, bg, g["scale"])
    for name, got, want in (("O", out_m, out), ("lse", lse_m, lse), ("O nshd", t(out_s), out),
                            ("gated", gated_m, gated)):
        assert torch.equal(got.reshape(reps, *want.shape), want.expand(reps, *want.shape)), name


@pytest.mark.parametrize("sk", [1023, 1022, 131])
def test_attention_fwd_picks_any_key(cuda, sk):
    """A bias that leaves one key's weight (exp(-300) for the others is below float32's smallest
    number): every row is that key's V, exactly, for keys at the edges of 64-key tiles that start
    at key 0 or -1 and of the groups of tiles whose mask bytes one lane loads."""
    n, h, sq, d = 2, 2, 131, 32
    inp = attention_inputs(n, h, sq, sk, d, torch.bfloat16, seed=sk, with_dout=False)
    g = {k: (v.to(cuda) if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    km = torch.ones((n, sk), dtype=torch.uint8, device=cuda)
    for key in (0, 62, 63, 64, 127, 128, 254, 255, 256, 511, 512, 767, 768, sk - 2, sk - 1):
        if key >= sk:
            continue
        bias = torch.full((h, sq, sk), -300.0, dtype=torch.bfloat16, device=cuda)
        bias[:, :, key] = 0.0
        out, _ = ops.attention_fwd(g["q"], g["k"], g["v"], bias, km, g["scale"])
        want = g["v"][:, :, key:key + 1].expand_as(out)
        assert torch.equal(out, want), key


# (dtype, scale, q, k): scales whose inverse two values of the type hold to 3e-7 (bfloat16, head
# dims 8 and 32), to 7e-6, or not at all (float16), and one dominating q.k of about 600 / scale.
SCALES = [(torch.bfloat16, 32 ** -0.5, 64.0, 56.0), (torch.bfloat16, 0.4989, 32.0, 40.0),
          (torch.bfloat16, 0.3, 32.0, 64.0), (torch.bfloat16, 0.25, 64.0, 40.0),
          (torch.bfloat16, 3e4, 0.125, 0.15625), (torch.float16, 32 ** -0.5, 64.0, 56.0),
          (torch.float16, 100.0, 2.0, 3.0), (torch.float16, 1e5, 0.0625, 0.09375),
          (torch.float16, 1e8, 2.0 ** -9, 1.5 * 2.0 ** -9)]


@pytest.mark.parametrize("sk", [64, 66, 67])
@pytest.mark.parametrize("dtype,scale,qv,kv", SCALES, ids=lambda v: str(v).replace("torch.", ""))
def test_attention_fwd_logits_are_float32(cuda, dtype, scale, qv, kv, sk):
    """A row with one key far above the others has that key's logit as its lse: scale * q.k and
    the bias both enter it as float32 values. The bound is eight roundings of 2^-24: the constants
    of the score's unit and of the two logarithms, the products and the sums. (At a multiple of
    eight keys only q.k is held to it.)"""
    n, h, sq, d = 1, 2, 6, 32
    q = torch.zeros((n, h, sq, d), dtype=dtype)
    k = torch.zeros((n, h, sk, d), dtype=dtype)
    v = torch.ones((n, h, sk, d), dtype=dtype)
    bias = torch.zeros((h, sq, sk), dtype=dtype)
    q[:, :, :3, 1] = qv
    k[:, :, sk - 1, 1] = kv
    bias[:, 3:, 5] = 600.0
    args = [t.to(cuda) for t in (q, k, v, bias)]
    _, lse = ops.attention_fwd(*args, None, scale)
    s32 = float(np.float32(scale))
    want = torch.tensor([qv * kv * s32] * 3 + [600.0] * 3, dtype=torch.float64)
    err = ((lse.cpu().double() - want) / want).abs().amax((0, 1))
    print("relative", err.tolist())
    held = err if sk % 8 else err[:3]
    assert (held <= 8 * 2.0 ** -24).all(), held.tolist()


@pytest.mark.parametrize("masked", [False, True])
def test_attention_fwd_without_keys(cuda, masked):
    """No keys at all (the C entries take such a call): O = 0 and lse = +inf, ungated in both
    layouts and gated, in the neighbourhood of an ordinary call on the same stream."""
    n, h, sq, d, c = 300, 4, 130, 32, 64
    inp = attention_inputs(n, h, sq, 64, d, torch.bfloat16, seed=3, with_dout=False)
    g = {k: (v.to(cuda) if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    x, wg, bg = (t.to(cuda) for t in gate_inputs(n, sq, c, h * d, torch.bfloat16, seed=4))
    lib, stream = _native.lib(), torch.cuda.current_stream().cuda_stream
    ptr = lambda t: t.data_ptr()  # noqa: E731
    km = ptr(g["kmask"]) if masked else None
    want = ops.attention(g["q"], g["k"], g["v"], g["bias"], None, g["scale"])
    for entry in ("plain", "nshd", "gated"):
        out = torch.full_like(g["q"], 7.0)
        gated = torch.full((n, sq, h * d), 7.0, dtype=out.dtype, device=cuda)
        lse = torch.zeros((n, h, sq), device=cuda)
        head = (stream, _native.BF16, ptr(g["q"]), ptr(g["k"]), ptr(g["v"]), ptr(g["bias"]), km)
        if entry == "plain":
            status = lib.clk_attention_fwd(*head, ptr(out), ptr(lse), n, h, sq, 0, d, 0.125, 64, 64)
        elif entry == "nshd":
            status = lib.clk_attention_fwd_nshd(*head, ptr(out), ptr(lse), n, h, sq, 0, d, 0.125)
        else:
            status = lib.clk_attention_fwd_gated(*head, ptr(x), ptr(wg), ptr(bg), ptr(gated),
                                                 ptr(out), ptr(lse), n, h, sq, 0, d, c, 0.125)
            assert not gated.any()
        assert status == _native.OK, _native.last_error()
        after = ops.attention(g["q"], g["k"], g["v"], g["bias"], None, g["scale"])
        assert not out.any() and bool((lse == np.inf).all())
        assert torch.equal(after, want)


# Key counts: odd, even and multiples of 8, with a ragged last tile or without.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=dname)
@pytest.mark.parametrize("sk,d", [(67, 32), (203, 32), (130, 16), (200, 32), (192, 64), (301, 8)])
def test_attention_fwd_infinite_bias(cuda, sk, d, dtype):
    """-inf in the bias is a weight of exactly 0: at single present keys, at all keys but one of a
    query, at absent keys, and (O = 0, lse = +inf) at all keys of a query. Forward in both layouts
    and gated, and the gradients; the queries around them are untouched."""
    n, h, sq, c = 3, 2, 131, 64
    inp = attention_inputs(n, h, sq, sk, d, dtype, seed=sk + d, masked_tail=0.1, masked_rows=1)
    gen = torch.Generator().manual_seed(sk)
    hole = torch.rand((h, sq, sk), generator=gen) < 0.3
    hole[:, :, 1] = False
    hole[:, 3::7] = False
    hole[0, 20] = True
    hole[0, 20, 1] = False
    nothing = (1, 64)  # the query without any key
    hole[nothing] = True
    inp["bias"] = inp["bias"].masked_fill(hole, -np.inf)
    g = {k: (v.to(cuda) if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    args = (g["q"], g["k"], g["v"], g["bias"], g["kmask"])
    out, lse = ops.attention_fwd(*args, g["scale"])
    full = (inp["kmask"] != 0).any(1)  # rows with a present key
    assert not out[full][:, nothing[0], nothing[1]].any()
    assert bool((lse[full][:, nothing[0], nothing[1]] == np.inf).all())
    # The oracle's masked logit would be that query's largest: the same value at every key there.
    safe = inp["bias"].clone()
    safe[nothing] = 0
    dout = g["dout"].clone()
    dout[:, nothing[0], nothing[1]] = 0
    o_ref, lse_ref = _oracle({**inp, "bias": safe})
    for t in (out, lse):
        t[full.to(cuda), nothing[0], nothing[1]] = 0
    o_ref[full.numpy(), nothing[0], nothing[1]] = 0
    lse_ref[full.numpy(), nothing[0], nothing[1]] = 0
    assert_close("O", out, o_ref, TOL[dname(dtype)]["o"])
    assert np.abs(np64(lse) - np.where(full.numpy()[:, None, None], lse_ref, np.log(sk))).max() < 5e-2
    t = lambda a: a.transpose(1, 2).contiguous()  # noqa: E731
    out_s = t(ops.attention_nshd(t(g["q"]), t(g["k"]), t(g["v"]), *args[3:], g["scale"])[0])
    assert torch.equal(out_s, out)
    x, wg, bg = (a.to(cuda) for a in gate_inputs(n, sq, c, h * d, dtype, seed=sk))
    gated = ops.attention_gated(*args, x, wg, bg, g["scale"])
    assert_close("gated", gated, ref_gate.attention_gate(o_ref, np64(x), np64(wg), np64(bg)),
                 TOL[dname(dtype)]["o"])
    out, lse = ops.attention_fwd(*args, g["scale"])
    grads = ops.attention_bwd(*args, out, dout, lse, g["scale"])
    refs = ref.attention_bwd(np64(inp["q"]), np64(inp["k"]), np64(inp["v"]), np64(safe),
                             inp["kmask"].numpy(), inp["scale"], np64(dout))
    for name, got, want in zip(("dQ", "dK", "dV", "dBias"), grads, refs):
        assert_close(name, got, want, TOL[dname(dtype)]["grad"])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=dname)
@pytest.mark.parametrize("value", [np.nan, np.inf, 3e4])
@pytest.mark.parametrize("sk", [67, 130, 200])
def test_attention_fwd_ignores_absent_keys_k(cuda, sk, value, dtype):
    """Whatever the K rows of absent keys hold (3e4 stands for 3e34 in bfloat16: q.k then passes
    the masked logit) reaches nothing, in the forms with and without the bias MFMA."""
    if value == 3e4 and dtype == torch.bfloat16:
        value = 3e34
    inp = attention_inputs(3, 2, 70, sk, 32, dtype, seed=sk, with_dout=False)
    inp["kmask"][0, 5] = inp["kmask"][1, sk - 1] = 0
    g = {k: (v.to(cuda) if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    g["k"][0, :, 5] = g["k"][1, 1, sk - 1] = value
    for sign in (1, -1):
        inp["scale"] *= sign
        out, lse = ops.attention_fwd(g["q"], g["k"], g["v"], g["bias"], g["kmask"], inp["scale"])
        o_ref, lse_ref = _oracle(inp)
        assert_close("O", out, o_ref, TOL[dname(dtype)]["o"])
        assert np.abs(np64(lse) - lse_ref).max() < 5e-2


@pytest.mark.parametrize("scale", [32 ** -0.5, -32 ** -0.5])
@pytest.mark.parametrize("sk", [66, 67, 200, 203])
def test_attention_fwd_lowest_float16_bias(cuda, sk, scale):
    """Float16 queries whose bias is the type's lowest value at every key (padded queries under an
    additive mask): no weight goes to absent keys (-1e9) or past the last one. The logits are near
    65504, where float32 steps by 2^-8: four roundings move a logit by 2^-7 and a weight by 0.8%."""
    n, h, sq, d = 3, 2, 70, 32
    inp = attention_inputs(n, h, sq, sk, d, torch.float16, seed=sk, masked_tail=0.2, masked_rows=1)
    inp["scale"] = scale
    inp["bias"][0, 3:40] = -65504.0
    inp["bias"][1, 60:] = -65504.0
    g = {k: (v.to(cuda) if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    out, lse = ops.attention_fwd(g["q"], g["k"], g["v"], g["bias"], g["kmask"], g["scale"])
    o_ref, lse_ref = _oracle(inp)
    assert_close("O", out, o_ref, TOL["f16"]["o"] + 0.008)
    full = (inp["kmask"] != 0).any(1).numpy()[:, None, None]
    assert np.abs(np64(lse) - np.where(full, lse_ref, np.log(sk))).max() <= 2.0 ** -6
    # The gradients recompute such a weight from its logit and lse: twice that error.
    grads = ops.attention_bwd(g["q"], g["k"], g["v"], g["bias"], g["kmask"], out, g["dout"], lse,
                              scale)
    refs = ref.attention_bwd(*(np64(inp[k]) for k in ("q", "k", "v", "bias")), inp["kmask"].numpy(),
                             scale, np64(inp["dout"]))
    for name, got, want in zip(("dQ", "dK", "dV", "dBias"), grads, refs):
        assert_close(name, got, want, TOL["f16"]["grad"] + 0.016)


# (N, H, Sq, Sk, D): one query and one key for 8.5 million (row, head) pairs, whose two parities of
# query blocks would pass the 2^32 - 1 threads of a launch, and 130 queries for 5.9 million, whose
# three 64-query blocks would.
@pytest.mark.parametrize("shape", [(65535, 130, 1, 1, 8), (65535, 90, 130, 2, 8)],
                         ids=lambda c: "x".join(map(str, c)))
def test_attention_fwd_most_blocks(cuda, shape):
    n, h, sq, sk, d = shape
    inp = attention_inputs(2, h, sq, sk, d, torch.bfloat16, seed=sq, with_dout=False)
    g = {k: (v.to(cuda) if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    q, k, v = (torch.zeros((n, *g[name].shape[1:]), dtype=torch.bfloat16, device=cuda)
               for name in "qkv")
    for big, name in ((q, "q"), (k, "k"), (v, "v")):
        big[0], big[-1] = g[name][0], g[name][1]
    out = ops.attention(q, k, v, g["bias"], None, g["scale"])
    assert_close("O", out[[0, -1]], _oracle(inp)[0], TOL["bf16"]["o"])
    assert not out[1:-1].any()
