"""LTX-2's attention prologue (full-row RMSNorm with an f32 weight, then the interleaved or the split rotation with
per-batch, per-head tables) through the C ABI, against the CPU oracle.  Same bars as the Wan / Flux prologue."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import bits_to_dev, err_stats, golden, to_dev_bf16, to_np
from maxdiffusion_amd import attention_op, ops

pytestmark = pytest.mark.gpu
MAX_ABS, MEAN_ABS = 2e-2, 2e-3


def _assert_close(got, ref, what):
  mx, mean = err_stats(got, ref)
  print(f"{what}: max-abs {mx:.3e} mean-abs {mean:.3e}", flush=True)
  assert mx <= 1.6e-2 and mean <= MEAN_ABS, what  # one bf16 rounding of |y| < 8


def _tables(rng, B, S, H, D, mode):
  if mode == "interleaved":  # attention_ltx2.py:292-295: [B,S,H*D], every angle repeated for its pair
    ang = rng.uniform(-3.1, 3.1, (B, S, H * D // 2))
    return np.repeat(np.cos(ang), 2, -1).astype(np.float32), np.repeat(np.sin(ang), 2, -1).astype(np.float32)
  ang = rng.uniform(-3.1, 3.1, (B, H, S, D // 2))  # :323-324
  return np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)


@pytest.mark.parametrize("H,D", [(32, 128), (32, 64), (5, 64), (48, 128)])
@pytest.mark.parametrize("mode", ["none", "interleaved", "split"])
@pytest.mark.parametrize("f32_in", [False, True])
def test_rows_against_oracle(dev, H, D, mode, f32_in):
  rng = np.random.default_rng(21)
  B, S = 2, 37
  x = rng.standard_normal((B, S, H * D)).astype(np.float32)
  if not f32_in:
    x = O.bf16_round(x)
  w = (1 + 0.1 * rng.standard_normal(H * D)).astype(np.float32)
  cos = sin = None
  if mode != "none":
    cos, sin = _tables(rng, B, S, H, D, mode)
  ref = O.norm_rope_ltx2(x, w, cos, sin, mode)
  xd = torch.from_numpy(x).to(dev) if f32_in else to_dev_bf16(x, dev)
  t = lambda a: None if a is None else torch.from_numpy(a).to(dev)
  for layout in ("bshd", "bhsd"):
    out = ops.norm_rope_rows(xd, t(w), t(cos), t(sin), heads=H, mode=mode, out_layout=layout)
    assert out.shape == (B, S, H, D) and out.dtype == torch.bfloat16
    _assert_close(to_np(out).reshape(B, S, H * D), ref, f"ltx2 {mode} H={H} D={D} f32_in={f32_in} {layout}")


def test_call_flow_of_the_attention_module(dev):
  # attention_ltx2.py:566-585: q gets rotary_emb; k gets k_rotary_emb, else rotary_emb for self-attention, else nothing
  rng = np.random.default_rng(22)
  B, Sq, Sk, H, D = 1, 20, 12, 4, 64
  q = rng.standard_normal((B, Sq, H * D)).astype(np.float32)
  k_self = rng.standard_normal((B, Sq, H * D)).astype(np.float32)
  k_cross = rng.standard_normal((B, Sk, H * D)).astype(np.float32)
  wq, wk = (1 + 0.1 * rng.standard_normal(H * D)).astype(np.float32), (1 + 0.1 * rng.standard_normal(H * D)).astype(np.float32)
  t = lambda a: torch.from_numpy(a).to(dev)
  for mode in ("interleaved", "split"):
    tab_q, tab_k = _tables(rng, B, Sq, H, D, mode), _tables(rng, B, Sk, H, D, mode)
    emb_q, emb_k = tuple(t(a) for a in tab_q), tuple(t(a) for a in tab_k)
    qo, ko = attention_op.hip_norm_rope_ltx2(t(q), t(k_self), t(wq), t(wk), H, rotary_emb=emb_q, rope_type=mode)
    _assert_close(to_np(qo).reshape(B, Sq, -1), O.norm_rope_ltx2(q, wq, *tab_q, mode), f"{mode} self q")
    _assert_close(to_np(ko).reshape(B, Sq, -1), O.norm_rope_ltx2(k_self, wk, *tab_q, mode), f"{mode} self k")
    qo, ko = attention_op.hip_norm_rope_ltx2(t(q), t(k_cross), t(wq), t(wk), H, rotary_emb=emb_q, rope_type=mode, is_self_attention=False)
    _assert_close(to_np(ko).reshape(B, Sk, -1), O.norm_rope_ltx2(k_cross, wk, None, None, "none"), f"{mode} cross k: norm only")
    qo, ko = attention_op.hip_norm_rope_ltx2(t(q), t(k_cross), t(wq), t(wk), H, rotary_emb=emb_q, k_rotary_emb=emb_k, rope_type=mode,
                                            is_self_attention=False)
    _assert_close(to_np(ko).reshape(B, Sk, -1), O.norm_rope_ltx2(k_cross, wk, *tab_k, mode), f"{mode} cross k with its own table")
    # q_mul (softmax scale carried by the prologue) goes into the f32 query scale: q scaled, k untouched
    m = ops.folded_q_mul(D)
    qo, ko = attention_op.hip_norm_rope_ltx2(t(q), t(k_self), t(wq), t(wk), H, rotary_emb=emb_q, rope_type=mode, q_mul=m)
    _assert_close(to_np(qo).reshape(B, Sq, -1) / m, O.norm_rope_ltx2(q, wq, *tab_q, mode), f"{mode} self q with q_mul")
    _assert_close(to_np(ko).reshape(B, Sq, -1), O.norm_rope_ltx2(k_self, wk, *tab_q, mode), f"{mode} self k with q_mul")
  with pytest.raises(ValueError, match="not supported"):
    attention_op.hip_norm_rope_ltx2(t(q), None, t(wq), t(wk), H, rope_type="rotate_half")


def test_golden_ltx2(dev):
  g = golden("norm_rope_ltx2.npz")
  x, H = bits_to_dev(g["x"], dev), int(g["heads"])
  t = lambda a: torch.from_numpy(a).to(dev)
  B, S, N = x.shape
  for mode, cs in (("none", (None, None)), ("interleaved", (g["cos_i"], g["sin_i"])), ("split", (g["cos_s"], g["sin_s"]))):
    cos, sin = (None if a is None else t(a) for a in cs)
    out = ops.norm_rope_rows(x, t(g["w"]), cos, sin, heads=H, mode=mode)
    _assert_close(to_np(out).reshape(B, S, N), g[f"out_{mode}"], f"ltx2 golden {mode}")


@pytest.mark.parametrize("mode,dtype", [("interleaved", torch.float32), ("split", torch.bfloat16), ("none", torch.float32)])
@pytest.mark.parametrize("H,D,S", [(3, 64, 37), (32, 64, 5), (32, 128, 9)])
def test_q_and_k_in_one_launch_equal_two_calls(dev, mode, dtype, H, D, S):
  """Self-attention's q and k go through one launch (shared tables, the query factor in the kernel): outputs and gradients
  equal, bit for bit, those of one call per tensor with the factor multiplied into the weight; partly filled workgroups."""
  from maxdiffusion_amd import attention_op as A
  B, N = 2, H * D
  gen = torch.Generator(device=dev).manual_seed(N + S)
  q, k = (torch.randn((B, S, N), generator=gen, device=dev).to(dtype).requires_grad_(True) for _ in range(2))
  wq, wk = ((1 + 0.1 * torch.randn(N, generator=gen, device=dev)).requires_grad_(True) for _ in range(2))
  ang = torch.rand((B, S, N) if mode == "interleaved" else (B, H, S, D // 2), generator=gen, device=dev) * 6.28
  tab = None if mode == "none" else (torch.cos(ang), torch.sin(ang))
  g = [torch.randn((B, S, H, D), generator=gen, device=dev).to(torch.bfloat16) for _ in range(2)]
  out = A.hip_norm_rope_ltx2(q, k, wq, wk, H, rotary_emb=tab, rope_type="interleaved" if mode == "none" else mode, q_mul=0.37)
  got = torch.autograd.grad(out, (q, k, wq, wk), g)
  f = torch.tensor(0.37, device=dev)
  cs = (None, None) if tab is None else tab
  want = (ops.norm_rope_rows(q.detach(), wq.detach() * f, *cs, heads=H, mode=mode), ops.norm_rope_rows(k.detach(), wk.detach(), *cs, heads=H, mode=mode))
  dq, dwq = ops.norm_rope_rows_backward(q.detach(), wq.detach() * f, g[0], *cs, heads=H, mode=mode)
  dk, dwk = ops.norm_rope_rows_backward(k.detach(), wk.detach(), g[1], *cs, heads=H, mode=mode)
  assert torch.equal(out[0], want[0]) and torch.equal(out[1], want[1])
  assert torch.equal(got[0], dq) and torch.equal(got[1], dk)
  # the partial sums are the same; the factor meets them before the second stage instead of after it
  assert torch.allclose(got[2], dwq * f, rtol=2e-6, atol=1e-6 * float(dwq.abs().max())) and torch.equal(got[3], dwk)
