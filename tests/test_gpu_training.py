"""Training reaches the HIP kernels: loss = sum(apply_attention(hip_norm_rope(...)) * g) differentiated by torch autograd
end to end -- prologue backward, attention backward -- against an f64 autograd reference built from library routines
(torch.nn.functional.rms_norm, a complex-multiply rotation, scaled_dot_product_attention) on the CPU.

The reference's trainer differentiates straight through `apply_attention` and the inline norm + rope
(trainers/wan_trainer.py:169, models/attention_flax.py:2655-2677); here the registry entry `hip_flash` and the prologue
hooks carry their own backward.  Bars: every tensor on the HIP path is bf16 between kernels (q, k, out, dq, dk, dx), so
gradients are held to rel-L2 <= 1e-2 and cosine >= 0.9999 of the f64 reference (measured: 3e-3 .. 4.5e-3)."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import cosine, rel_l2, to_dev_bf16
from maxdiffusion_amd import _lib
from maxdiffusion_amd import attention_op as A
from maxdiffusion_amd import ops

pytestmark = pytest.mark.gpu


def _leaf(x, dev, dtype=torch.bfloat16):
  t = to_dev_bf16(x, dev) if dtype == torch.bfloat16 else torch.from_numpy(x).to(dev)
  return t.requires_grad_(True)


def _rope_complex(y, cos, sin):
  yc = torch.view_as_complex(y.reshape(*y.shape[:-1], -1, 2))
  rot = torch.complex(torch.tensor(cos, dtype=torch.float64), torch.tensor(sin, dtype=torch.float64))[None, :, None, :]
  return torch.view_as_real(yc * rot).reshape(y.shape)


def _check(got, ref, what):
  g, r = got.detach().float().cpu().numpy(), ref.detach().numpy()
  rl, cs = rel_l2(g, r), cosine(g, r)
  print(f"{what}: rel-l2 {rl:.3e} cosine {cs:.6f}", flush=True)
  assert rl <= 1e-2 and cs >= 0.9999, what


@pytest.mark.parametrize("rank4,masked", [(True, False), (False, True)])
def test_wan_prologue_and_attention_end_to_end(dev, rank4, masked):
  B, H, D, grid = 2, 3, 128, (2, 5, 9)
  S, N = grid[0] * grid[1] * grid[2], 3 * 128
  scale = D**-0.5
  xq, xk, xv = O.normal_bf16((B, S, N), 0), O.normal_bf16((B, S, N), 1), O.normal_bf16((B, S, N), 2)
  wq, wk = O.norm_weight(N, 3), O.norm_weight(N, 4)
  g = O.normal_bf16((B, S, N), 5)
  cos, sin = O.wan_rope_table(grid, D)
  keep = np.ones((B, S), bool)
  if masked:
    keep[0, 40:] = False
    keep[1, ::3] = False

  q, k, v, tq, tk = (_leaf(x, dev) for x in (xq, xk, xv, wq, wk))
  freqs = torch.complex(torch.from_numpy(cos), torch.from_numpy(sin)).to(dev)[None, None]  # as WanRotaryPosEmbed returns it
  qn, kn = A.hip_norm_rope(q, k, tq, tk, freqs, H, out_layout="bhsd" if rank4 else "bshd")
  assert qn.requires_grad and kn.requires_grad
  op = A.AttentionOp(attention_kernel="hip_flash", scale=scale, heads=H, dim_head=D, residual_checkpoint_name="attn_out")
  if rank4:  # FlaxWanAttention hands [B,H,S,D] (attention_flax.py:2673-2677)
    out = op.apply_attention(qn.permute(0, 2, 1, 3), kn.permute(0, 2, 1, 3), v.view(B, S, H, D).permute(0, 2, 1, 3))
  else:
    out = op.apply_attention(qn.reshape(B, S, N), kn.reshape(B, S, N), v, attention_mask=torch.from_numpy(keep).to(dev) if masked else None)
  assert out.shape == (B, S, N) and out.requires_grad
  (out.float() * to_dev_bf16(g, dev).float()).sum().backward()

  rq, rk, rv, rwq, rwk = (torch.tensor(x, dtype=torch.float64, requires_grad=True) for x in (xq, xk, xv, wq, wk))
  yq = _rope_complex(torch.nn.functional.rms_norm(rq, (N,), rwq, eps=1e-6).reshape(B, S, H, D), cos, sin).transpose(1, 2)
  yk = _rope_complex(torch.nn.functional.rms_norm(rk, (N,), rwk, eps=1e-6).reshape(B, S, H, D), cos, sin).transpose(1, 2)
  am = torch.from_numpy(keep)[:, None, None, :] if (masked and not rank4) else None
  ro = torch.nn.functional.scaled_dot_product_attention(yq, yk, rv.reshape(B, S, H, D).transpose(1, 2), attn_mask=am, scale=scale)
  (ro.transpose(1, 2).reshape(B, S, N) * torch.tensor(g, dtype=torch.float64)).sum().backward()
  _check(out, ro.transpose(1, 2).reshape(B, S, N), "forward")
  for got, ref, name in ((q, rq, "d q_in"), (k, rk, "d k_in"), (v, rv, "d v"), (tq, rwq, "d wq"), (tk, rwk, "d wk")):
    assert got.grad is not None and got.grad.dtype == got.dtype and got.grad.shape == got.shape
    _check(got.grad, ref.grad, name)
  if masked and not rank4:  # masked keys receive no gradient through the attention
    assert not v.grad[0, 40:].any()


@pytest.mark.parametrize("with_bias", [True, False])
def test_fused_projection_prologue_and_attention_end_to_end(dev, with_bias):
  """One fused q|k|v projection output [B,S,3*H*D] (the three Linears of attention_flax.py:2653-2663 as one GEMM, their
  biases added by the prologue): gradients for the fused buffer, the biases and the norm weights."""
  B, H, D, grid = 2, 3, 128, (2, 5, 9)
  S, N = grid[0] * grid[1] * grid[2], 3 * 128
  scale = D**-0.5
  xqkv = O.normal_bf16((B, S, 3 * N), 0)
  xb = (0.5 * O.normal_bf16((3 * N,), 1)).astype(np.float32)
  wq, wk = O.norm_weight(N, 3), O.norm_weight(N, 4)
  g = O.normal_bf16((B, S, N), 5)
  cos, sin = O.wan_rope_table(grid, D)

  qkv, tq, tk = (_leaf(x, dev) for x in (xqkv, wq, wk))
  tb = _leaf(xb, dev) if with_bias else None
  freqs = torch.complex(torch.from_numpy(cos), torch.from_numpy(sin)).to(dev)[None, None]
  qn, kn, vn = A.hip_norm_rope_qkv(qkv, tq, tk, freqs, H, bias=tb)
  assert qn.requires_grad and kn.requires_grad and vn.requires_grad
  op = A.AttentionOp(attention_kernel="hip_flash", scale=scale, heads=H, dim_head=D)
  out = op.apply_attention(qn.permute(0, 2, 1, 3), kn.permute(0, 2, 1, 3), vn.permute(0, 2, 1, 3))
  (out.float() * to_dev_bf16(g, dev).float()).sum().backward()
  with pytest.raises(ValueError, match="inplace"):
    A.hip_norm_rope_qkv(qkv, tq, tk, freqs, H, bias=tb, inplace=True)

  rqkv, rwq, rwk = (torch.tensor(x, dtype=torch.float64, requires_grad=True) for x in (xqkv, wq, wk))
  xb16 = to_dev_bf16(xb, "cpu").double().numpy() if with_bias else np.zeros(3 * N)  # the bias as the kernel sees it: bf16
  rb = torch.tensor(xb16, dtype=torch.float64, requires_grad=True)
  u = rqkv + rb
  yq = _rope_complex(torch.nn.functional.rms_norm(u[..., :N], (N,), rwq, eps=1e-6).reshape(B, S, H, D), cos, sin).transpose(1, 2)
  yk = _rope_complex(torch.nn.functional.rms_norm(u[..., N:2 * N], (N,), rwk, eps=1e-6).reshape(B, S, H, D), cos, sin).transpose(1, 2)
  ro = torch.nn.functional.scaled_dot_product_attention(yq, yk, u[..., 2 * N:].reshape(B, S, H, D).transpose(1, 2), scale=scale)
  ro = ro.transpose(1, 2).reshape(B, S, N)
  (ro * torch.tensor(g, dtype=torch.float64)).sum().backward()
  _check(out, ro, "forward")
  checks = [(qkv, rqkv, "d qkv"), (tq, rwq, "d wq"), (tk, rwk, "d wk")] + ([(tb, rb, "d bias")] if with_bias else [])
  for got, ref, name in checks:
    assert got.grad is not None and got.grad.dtype == got.dtype and got.grad.shape == got.shape
    _check(got.grad, ref.grad, name)
  for blk, name in ((slice(0, N), "q"), (slice(N, 2 * N), "k"), (slice(2 * N, 3 * N), "v")):  # each column block on its own
    _check(qkv.grad[..., blk], rqkv.grad[..., blk], "d qkv block " + name)


def test_flux_prologue_and_attention_end_to_end(dev):
  B, H, D, n_txt = 1, 4, 128, 7
  ids = O.flux_ids(n_txt, 5, 6)
  L = ids.shape[0]
  scale = D**-0.5
  xq, xk, xv = (O.normal_bf16((B, L, H, D), s) for s in (0, 1, 2))
  ws = [O.norm_weight(D, s) for s in (3, 4, 5, 6)]
  g = O.normal_bf16((B, L, H * D), 7)
  cos, sin = O.flux_rope_table(ids)
  q, k, v = (_leaf(x, dev) for x in (xq, xk, xv))
  tw = [_leaf(w, dev) for w in ws]
  qn, kn = A.hip_norm_rope(q, k, tw[0], tw[1], (torch.from_numpy(cos).to(dev), torch.from_numpy(sin).to(dev)), H, per_head=True,
                           wq_txt=tw[2], wk_txt=tw[3], n_txt=n_txt)
  op = A.AttentionOp(attention_kernel="hip_flash", scale=scale, heads=H, dim_head=D)
  out = op.apply_attention(qn.reshape(B, L, H * D), kn.reshape(B, L, H * D), v.reshape(B, L, H * D))
  (out.float() * to_dev_bf16(g, dev).float()).sum().backward()

  rq, rk, rv = (torch.tensor(x, dtype=torch.float64, requires_grad=True) for x in (xq, xk, xv))
  rw = [torch.tensor(w, dtype=torch.float64, requires_grad=True) for w in ws]
  norm = lambda x, w_img, w_txt: torch.cat([torch.nn.functional.rms_norm(x[:, :n_txt], (D,), w_txt, eps=1e-6),
                                            torch.nn.functional.rms_norm(x[:, n_txt:], (D,), w_img, eps=1e-6)], dim=1)
  yq = _rope_complex(norm(rq, rw[0], rw[2]), cos, sin).transpose(1, 2)
  yk = _rope_complex(norm(rk, rw[1], rw[3]), cos, sin).transpose(1, 2)
  ro = torch.nn.functional.scaled_dot_product_attention(yq, yk, rv.transpose(1, 2), scale=scale).transpose(1, 2).reshape(B, L, H * D)
  (ro * torch.tensor(g, dtype=torch.float64)).sum().backward()
  _check(out, ro, "forward")
  for got, ref, name in ((q, rq, "d q"), (k, rk, "d k"), (v, rv, "d v"), (tw[0], rw[0], "d wq"), (tw[1], rw[1], "d wk"),
                         (tw[2], rw[2], "d wq_txt"), (tw[3], rw[3], "d wk_txt")):
    _check(got.grad, ref.grad, name)


@pytest.mark.parametrize("rope_type", ["interleaved", "split"])
def test_ltx2_prologue_and_attention_end_to_end(dev, rope_type):
  """LTX-2: f32 activations and f32 norm weights (attention_ltx2.py:415-432), head dim 64, per-head tables."""
  B, S, H, D = 2, 50, 4, 64
  N = H * D
  scale = D**-0.5
  rng = np.random.default_rng(3)
  xq, xk, xv = (rng.standard_normal((B, S, N)).astype(np.float32) for _ in range(3))
  wq, wk = (1 + 0.1 * rng.standard_normal(N)).astype(np.float32), (1 + 0.1 * rng.standard_normal(N)).astype(np.float32)
  g = O.normal_bf16((B, S, N), 7)
  if rope_type == "interleaved":
    ang = rng.uniform(-3, 3, (B, S, N // 2))
    cos, sin = np.repeat(np.cos(ang), 2, -1).astype(np.float32), np.repeat(np.sin(ang), 2, -1).astype(np.float32)
  else:
    ang = rng.uniform(-3, 3, (B, H, S, D // 2))
    cos, sin = np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)
  q, k, v, tq, tk = (_leaf(x, dev, torch.float32) for x in (xq, xk, xv, wq, wk))
  tabs = (torch.from_numpy(cos).to(dev), torch.from_numpy(sin).to(dev))
  qn, kn = A.hip_norm_rope_ltx2(q, k, tq, tk, H, rotary_emb=tabs, rope_type=rope_type)
  op = A.AttentionOp(attention_kernel="hip_flash", scale=scale, heads=H, dim_head=D)
  out = op.apply_attention(qn.reshape(B, S, N), kn.reshape(B, S, N), v)
  assert out.dtype == torch.bfloat16  # q, k come out of the prologue as bf16; v is cast by the registry entry
  (out.float() * to_dev_bf16(g, dev).float()).sum().backward()

  rq, rk, rv, rwq, rwk = (torch.tensor(x, dtype=torch.float64, requires_grad=True) for x in (xq, xk, xv, wq, wk))
  c, s_ = torch.tensor(cos, dtype=torch.float64), torch.tensor(sin, dtype=torch.float64)

  def rot(y):
    if rope_type == "interleaved":
      yr = y.reshape(B, S, N // 2, 2)
      return y * c + torch.stack([-yr[..., 1], yr[..., 0]], dim=-1).reshape(B, S, N) * s_
    yh = y.reshape(B, S, H, 2, D // 2).permute(0, 2, 1, 3, 4)
    a1, a2 = yh[..., 0, :], yh[..., 1, :]
    return torch.stack([a1 * c - a2 * s_, a2 * c + a1 * s_], dim=-2).permute(0, 2, 1, 3, 4).reshape(B, S, N)

  heads_first = lambda t: t.reshape(B, S, H, D).transpose(1, 2)
  yq, yk = rot(torch.nn.functional.rms_norm(rq, (N,), rwq, eps=1e-6)), rot(torch.nn.functional.rms_norm(rk, (N,), rwk, eps=1e-6))
  ro = torch.nn.functional.scaled_dot_product_attention(heads_first(yq), heads_first(yk), heads_first(rv), scale=scale)
  ro = ro.transpose(1, 2).reshape(B, S, N)
  (ro * torch.tensor(g, dtype=torch.float64)).sum().backward()
  _check(out, ro, "forward")
  for got, ref, name in ((q, rq, "d q_in"), (k, rk, "d k_in"), (v, rv, "d v"), (tq, rwq, "d wq"), (tk, rwk, "d wk")):
    assert got.grad.dtype == torch.float32
    _check(got.grad, ref.grad, name)


def test_no_grad_path_is_unchanged(dev):
  """Without autograd recording the registry entry and the hook call the plain operators (no lse, nothing saved)."""
  B, S, H, D = 1, 40, 2, 128
  q, k, v = (to_dev_bf16(O.normal_bf16((B, S, H * D), s), dev) for s in (0, 1, 2))
  op = A.AttentionOp(attention_kernel="hip_flash", scale=D**-0.5, heads=H, dim_head=D)
  plain = op.apply_attention(q, k, v)
  qg = q.clone().requires_grad_(True)
  with torch.no_grad():
    assert not op.apply_attention(qg, k, v).requires_grad
  tracked = op.apply_attention(qg, k, v)
  assert tracked.requires_grad and torch.equal(tracked.detach(), plain)


def test_saved_tensor_hooks_around_the_backward(dev):
  """What a hook hands back is used (a copy with the same layout, as an offloading hook returns it; a mask's tile lists do
  not pass through hooks) or refused with a ValueError (another dtype): never read as something it is not."""
  B, H, D, S = 1, 2, 128, 70
  N = H * D
  gen = torch.Generator(device=dev).manual_seed(3)
  mk = lambda *s, dt=torch.bfloat16: torch.randn(s, generator=gen, device=dev).to(dt).requires_grad_(True)
  g = torch.randn((B, S, N), generator=gen, device=dev).to(torch.bfloat16)
  keep = torch.arange(S, device=dev)[None] < 41
  op = A.AttentionOp(attention_kernel="hip_flash", scale=D**-0.5, heads=H, dim_head=D, dtype=torch.bfloat16)
  q, k, v, wq, wk = mk(B, S, N), mk(B, S, N), mk(B, S, N), mk(N), mk(N)
  qkv, bias = mk(B, S, 3 * N), mk(3 * N)
  hq, hk, hw = mk(B, S, H, D), mk(B, S, H, D), mk(D)
  rq, rk, rw = mk(B, S, N, dt=torch.float32), mk(B, S, N, dt=torch.float32), mk(N, dt=torch.float32)
  gh = g.view(B, S, H, D)
  freqs = torch.polar(torch.ones(S, D // 2, device=dev), torch.rand(S, D // 2, generator=gen, device=dev))[None, None]
  calls = {
      "attention": (lambda: (op.apply_attention(q, k, v, attention_mask=keep),), (q, k, v), (g,)),
      "full row": (lambda: A.hip_norm_rope(q, k, wq, wk, freqs, H), (q, k, wq, wk), (gh, gh)),
      "fused": (lambda: A.hip_norm_rope_qkv(qkv, wq, wk, freqs, H, bias=bias), (qkv, bias, wq, wk), (gh, gh, gh)),
      "per head": (lambda: A.hip_norm_rope(hq, hk, hw, hw, freqs, H, per_head=True), (hq, hk, hw), (gh, gh)),
      "rows": (lambda: A.hip_norm_rope_ltx2(rq, rk, rw, rw, H), (rq, rk, rw), (gh, gh)),
  }
  lossy = lambda t: t.to(torch.bfloat16) if t.dtype == torch.float32 else t.to(torch.float32)
  for name, (call, leaves, gs) in calls.items():
    print(name, flush=True)
    want = torch.autograd.grad(call(), leaves, gs)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.to(dev)):
      out = call()
    for a, b in zip(torch.autograd.grad(out, leaves, gs), want):
      assert torch.equal(a, b), name
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lossy):
      out = call()
    with pytest.raises(ValueError):
      torch.autograd.grad(out, leaves, gs)


@pytest.mark.parametrize("rank4", [False, True])
def test_unpadded_head_dim_at_any_address(dev, rank4):
  """A head dim that the kernels walk unpadded (80), with operands and an output gradient that start 2 bytes past an aligned
  address: taken as the padding copy takes them, and the same result as for aligned copies within two bf16 roundings
  (the padded kernels sum in another order)."""
  B, H, D, S = 1, 2, 80, 70
  N = H * D
  shape = (B, H, S, D) if rank4 else (B, S, N)
  gen = torch.Generator(device=dev).manual_seed(4)
  base = [torch.randn(B * S * N + 1, generator=gen, device=dev).to(torch.bfloat16) for _ in range(4)]
  odd = [t[1:].view(shape).requires_grad_(True) for t in base[:3]]
  even = [t.detach().clone().requires_grad_(True) for t in odd]
  g = base[3][1:].view(B, S, N)
  op = A.AttentionOp(attention_kernel="hip_flash", scale=D**-0.5, heads=H, dim_head=D, dtype=torch.bfloat16)
  want = op.apply_attention(*even)
  want_grads = torch.autograd.grad(want, even, g.clone())
  for leaves in (odd, even):  # operands and gradient at odd addresses, then the gradient alone
    out = op.apply_attention(*leaves)
    for a, b in zip((out, *torch.autograd.grad(out, leaves, g)), (want, *want_grads)):
      assert rel_l2(a.detach().float().cpu().numpy(), b.detach().float().cpu().numpy()) <= 8e-3


def _fused_prologue(dev, B, S, H, D, bias=True):
  """Leaves of the fused prologue and a call of it."""
  N = H * D
  gen = torch.Generator(device=dev).manual_seed(B + S + H)
  mk = lambda *s: torch.randn(s, generator=gen, device=dev).to(torch.bfloat16).requires_grad_(True)
  freqs = torch.polar(torch.ones(S, D // 2, device=dev), torch.rand(S, D // 2, generator=gen, device=dev))[None, None]
  leaves = (mk(B, S, 3 * N), mk(N), mk(N)) + ((mk(3 * N),) if bias else ())
  return leaves, lambda: A.hip_norm_rope_qkv(*leaves[:3], freqs, H, bias=leaves[3] if bias else None), gen


@pytest.mark.parametrize("gaps,at", [(8, 4), (0, 4), (24, 0)])
def test_value_gradient_at_any_address(dev, gaps, at):
  """The value block's gradient as a view that starts `at` columns into wider rows, next to gradients of q and k with the same
  strides: the result of dense copies, bit for bit (the same values in the same order)."""
  B, S, H, D = 2, 37, 3, 64
  leaves, call, gen = _fused_prologue(dev, B, S, H, D)
  wide = [torch.randn((B, S, H, D + gaps), generator=gen, device=dev).to(torch.bfloat16) for _ in range(2)]
  edge = torch.randn(B * S * H * (D + gaps) + 8, generator=gen, device=dev).to(torch.bfloat16)
  gq, gk = (t[..., :D] for t in wide)
  gv = edge.as_strided(gq.shape, gq.stride(), at)
  got = torch.autograd.grad(call(), leaves, (gq, gk, gv))
  want = torch.autograd.grad(call(), leaves, (gq.contiguous(), gk.contiguous(), gv.contiguous()))
  for a, b in zip(got, want):
    assert torch.equal(a, b)


@pytest.mark.parametrize("which", [(0, 1), (0,), (0, 2), (0, 1, 2)])
def test_expanded_output_gradients(dev, which):
  """Output gradients expanded over the batch (what a sum over it hands back) beside dense ones."""
  B, S, H, D = 2, 21, 2, 64
  leaves, call, gen = _fused_prologue(dev, B, S, H, D)
  mk = lambda b: torch.randn((b, S, H, D), generator=gen, device=dev).to(torch.bfloat16)
  gs = [mk(1).expand(B, S, H, D) if i in which else mk(B) for i in range(3)]
  got = torch.autograd.grad(call(), leaves, gs)
  want = torch.autograd.grad(call(), leaves, [g.contiguous() for g in gs])
  for a, b in zip(got, want):
    assert torch.equal(a, b)


@pytest.mark.parametrize("form,table", [(f, "complex") for f in ("full row", "fused", "fused, no bias", "slices")] +
                         [(f, t) for f in ("per head", "per head slices") for t in ("complex", "repeated", "matrix")])
def test_table_made_in_inference_mode_and_rewritten(dev, form, table):
  """The backward uses the table that the forward read: one made in inference mode (a cache that sampling filled) is taken,
  and one rewritten in between changes nothing.  `slices`: q and k as column blocks of one buffer, and the fused form
  without biases, which go through the Python nodes."""
  B, S, H, D = 1, 35, 2, 64
  N = H * D
  leaves, fused, gen = _fused_prologue(dev, B, S, H, D, bias=form != "fused, no bias")
  per_head = form.startswith("per head")
  ang = torch.rand(S, D // 2, generator=gen, device=dev)
  c, s = torch.cos(ang), torch.sin(ang)

  def make():
    if table == "complex":
      return (torch.polar(torch.ones_like(ang), ang)[None, None],)
    if table == "repeated":
      return c.repeat_interleave(2, 1), s.repeat_interleave(2, 1)
    return (torch.stack([torch.stack([c, -s], -1), torch.stack([s, c], -1)], -2),)

  qkv, wq, wk = leaves[:3]
  wide = qkv.detach()
  q, k = (wide[..., i * N:(i + 1) * N] for i in (0, 1))
  w = (wq, wk)
  if per_head:
    q, k = q.unflatten(2, (H, D)), k.unflatten(2, (H, D))
    w = tuple(t.detach()[:D].requires_grad_(True) for t in w)
  if "slices" not in form:
    q, k = q.contiguous(), k.contiguous()
  q, k = (t.detach().requires_grad_(True) for t in (q, k))

  def run(rewrite, make):
    t = make()
    f = t[0] if len(t) == 1 else t
    if form.startswith("fused"):
      x = leaves
      out = A.hip_norm_rope_qkv(qkv, wq, wk, f, H, bias=leaves[3] if len(leaves) == 4 else None)
    else:
      x = (q, k) + w
      out = A.hip_norm_rope(q, k, *w, f, H, per_head=per_head)
    if rewrite:
      for a in t:
        a.zero_()
    g = torch.ones((B, S, H, D), dtype=torch.bfloat16, device=dev)
    return torch.autograd.grad(out, x, (g,) * len(out))

  def sampled():
    with torch.inference_mode():
      return make()

  want = run(False, make)
  for got in (run(False, sampled), run(True, make)):
    for a, b in zip(got, want):
      assert torch.equal(a, b)


def _ltx2(dev):
  B, S, H, D = 1, 23, 2, 64
  gen = torch.Generator(device=dev).manual_seed(6)
  mk = lambda *s: torch.randn(s, generator=gen, device=dev).requires_grad_(True)
  g = torch.randn((B, S, H, D), generator=gen, device=dev).to(torch.bfloat16)
  return mk(B, S, H * D), mk(B, S, H * D), mk(H * D), mk(H * D), H, g


def test_ltx2_query_weight_under_a_factor(dev):
  """With q_mul the backward uses the query weight that the forward read: rewritten in between, or made in inference mode."""
  q, k, wq, wk, H, g = _ltx2(dev)
  want = torch.autograd.grad(A.hip_norm_rope_ltx2(q, k, wq, wk, H, q_mul=0.5), (q, k, wq, wk), (g, g))
  w = wq.detach().clone().requires_grad_(True)
  out = A.hip_norm_rope_ltx2(q, k, w, wk, H, q_mul=0.5)
  with torch.no_grad():
    w.zero_()
  for a, b in zip(torch.autograd.grad(out, (q, k, w, wk), (g, g)), want):
    assert torch.equal(a, b)
  with torch.inference_mode():
    w = wq.detach().clone()
  for a, b in zip(torch.autograd.grad(A.hip_norm_rope_ltx2(q, k, w, wk, H, q_mul=0.5), (q, k, wk), (g, g)), (want[0], want[1], want[3])):
    assert torch.equal(a, b)


def test_a_refused_training_call_raises_the_library_error(dev):
  """What a kernel refuses in training raises MdattnError with its code: in the forward as without gradients, and in the backward."""
  mk = lambda *s, dtype=torch.bfloat16: torch.ones(s, dtype=dtype, device=dev).requires_grad_(True)
  wide, small = mk(1, 4, 65 * 128), mk(1, 4, 2, 32)  # more than 8,192 channels; a head dim that the per-head kernels do not have
  calls = [lambda: A.hip_norm_rope(wide, None, mk(65 * 128), None, None, 65),
           lambda: A.hip_norm_rope_qkv(mk(1, 4, 3 * 65 * 128), mk(65 * 128), mk(65 * 128), None, 65, bias=mk(3 * 65 * 128)),
           lambda: A.hip_norm_rope(small, None, mk(32), None, None, 2, per_head=True),
           lambda: A.hip_norm_rope_ltx2(wide, None, mk(65 * 128, dtype=torch.float32), None, 65)]
  for call in calls:
    with torch.no_grad(), pytest.raises(_lib.MdattnError) as plain:
      call()
    with pytest.raises(_lib.MdattnError) as e:
      call()
    assert e.value.code == plain.value.code == -2

  q, k, v = (mk(1, 8, 2 * 128) for _ in range(3))
  off = torch.ones(8 * 256 + 8, dtype=torch.bfloat16, device=dev)[4:-4]  # 8 bytes off a 16-byte address
  op = A.AttentionOp(attention_kernel="hip_flash", heads=2, dim_head=128, scale=0.1)
  for out in (op.apply_attention(q, k, v), A.hip_norm_rope(q, None, mk(256), None, None, 2)[0]):
    with pytest.raises(_lib.MdattnError) as e:
      out.backward(off.view(out.shape))
    assert e.value.code == -3


@pytest.mark.parametrize("training", [False, True])
def test_a_table_and_a_weight_too_small_to_be_copied(dev, training):
  """Sizes that are no multiple of 16 bytes, which a training call's copies refuse: such a call ends as it does without them."""
  mk = lambda n, dtype=torch.bfloat16: torch.randn((1, 3, n), device=dev).to(dtype).requires_grad_(training)
  table = torch.polar(torch.ones((3, 1), device=dev), torch.rand((3, 1), device=dev))  # 24 bytes
  w = torch.ones(6, device=dev)
  for call in (lambda: A.hip_norm_rope(mk(4), mk(4), w[:4].bfloat16(), w[:4].bfloat16(), table, 2),
               lambda: A.hip_norm_rope_ltx2(mk(6, torch.float32), mk(6, torch.float32), w, w, 1, rotary_emb=None, q_mul=0.5)):
    with pytest.raises(_lib.MdattnError) as e:
      call()
    assert e.value.code == _lib.E_UNSUPPORTED


def test_ltx2_gradient_of_the_query_alone(dev):
  """A loss that reaches one of q and k leaves the other and its weight without a gradient, and operands that need none get none."""
  q, k, wq, wk, H, g = _ltx2(dev)
  both = torch.autograd.grad(A.hip_norm_rope_ltx2(q, k, wq, wk, H, q_mul=0.5), (q, k, wq, wk), (g, g))
  for i in (0, 1):
    got = torch.autograd.grad(A.hip_norm_rope_ltx2(q, k, wq, wk, H, q_mul=0.5)[i], (q, k, wq, wk), g, allow_unused=True)
    for j in range(4):
      assert torch.equal(got[j], both[j]) if j % 2 == i else got[j] is None
  qo, ko = A.hip_norm_rope_ltx2(q, k.detach(), wq, wk.detach(), H)
  assert qo.requires_grad and not ko.requires_grad
  qo, ko = A.hip_norm_rope_ltx2(q.detach(), k, wq.detach(), wk, H)
  assert ko.requires_grad and not qo.requires_grad


def test_ltx2_backward_through_the_query_then_the_key(dev):
  """Two losses with a backward each, as through two nodes: the second one takes what the first left, once, and refuses it when
  it was rewritten."""
  q, k, wq, wk, H, g = _ltx2(dev)
  both = torch.autograd.grad(A.hip_norm_rope_ltx2(q, k, wq, wk, H, q_mul=0.5), (q, k, wq, wk), (g, g))
  for order in ((0, 1), (1, 0)):
    out = A.hip_norm_rope_ltx2(q, k, wq, wk, H, q_mul=0.5)
    for i in order:
      for got, want in zip(torch.autograd.grad(out[i], (q, wq) if i == 0 else (k, wk), g), both[i::2]):
        assert torch.equal(got, want)
    for i in order:
      with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out[i], (q, wq) if i == 0 else (k, wk), g)
  out = A.hip_norm_rope_ltx2(q, k, wq, wk, H)
  torch.autograd.grad(out[0], q, g)
  with torch.no_grad():
    k.mul_(2)
  with pytest.raises(RuntimeError, match="inplace"):
    torch.autograd.grad(out[1], k, g)


@pytest.mark.parametrize("form", ["slices", "per head slices", "fused, no bias"])
def test_gradients_of_the_python_nodes(dev, form):
  """Calls that the C++ nodes leave to the Python ones -- q and k as column blocks of one buffer, the fused form without biases --
  against the dense call on the same values, with a table that is read in place.  The slices: the same kernels on the same
  values, bit for bit.  Without biases: the kernel without them against one that adds zeros, where sums may round in another
  order: half a unit in the last place of bf16 on either side, 2 * 2^-9."""
  B, S, H, D = 2, 37, 3, 64
  N = H * D
  per_head = form.startswith("per head")
  (qkv, wq, wk, bias), _, gen = _fused_prologue(dev, B, S, H, D)
  table = torch.polar(torch.ones(S, D // 2, device=dev), torch.rand(S, D // 2, generator=gen, device=dev))
  gs = [torch.randn((B, S, H, D), generator=gen, device=dev).to(torch.bfloat16) for _ in range(3)]
  if form == "fused, no bias":
    with torch.no_grad():
      bias.zero_()
    got = torch.autograd.grad(A.hip_norm_rope_qkv(qkv, wq, wk, table, H), (qkv, wq, wk), gs)
    want = torch.autograd.grad(A.hip_norm_rope_qkv(qkv, wq, wk, table, H, bias=bias), (qkv, wq, wk), gs)
    for a, b in zip(got, want):
      assert rel_l2(a.float().cpu().numpy(), b.float().cpu().numpy()) <= 2**-8
    return
  w = tuple(t.detach()[:D if per_head else N].clone().requires_grad_(True) for t in (wq, wk))
  cut = [qkv.detach()[..., i * N:(i + 1) * N] for i in (0, 1)]
  if per_head:
    cut = [t.unflatten(2, (H, D)) for t in cut]
  grads = []
  for q, k in (cut, [t.contiguous() for t in cut]):
    q, k = (t.detach().requires_grad_(True) for t in (q, k))
    grads.append(torch.autograd.grad(A.hip_norm_rope(q, k, *w, table, H, per_head=per_head), (q, k) + w, gs[:2]))
  for a, b in zip(*grads):
    assert torch.equal(a, b)
