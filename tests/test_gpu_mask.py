"""Key padding masks: `[B,Skv]` keep-masks through the additive-bias entry point (HIP, through the C ABI).

Oracle: dense softmax with the masked keys excluded; rows without a kept key return 0
(models/attention_flax.py:1552-1554).  Hand fixtures follow the reference's own mask tests
(tests/ltx2/test_attention_ltx2.py:38-116)."""
import ctypes
import math

import numpy as np
import pytest
import torch

import oracle as O
from helpers import err_stats, hsd, rel_l2, to_dev_bf16, to_np
from maxdiffusion_amd import attention_op, ops

pytestmark = pytest.mark.gpu
MAX_ABS, MEAN_ABS, LSE_ABS, REL_L2 = 2e-2, 2e-3, 1e-3, 1.5e-2


def test_mask_bias_kernel(dev):
  keep = torch.tensor([[1, 0, 1, 1, 0], [0, 0, 0, 0, 1]], dtype=torch.bool, device=dev)
  bias = ops.key_mask_bias(keep)
  assert bias.shape == (2, 32) and bias.dtype == torch.float32
  want = torch.full((2, 32), -math.inf)
  want[0, [0, 2, 3]] = 0.0
  want[1, 4] = 0.0
  assert torch.equal(bias.cpu(), want)
  assert torch.equal(ops.key_mask_bias(keep, masked_value=-10000.0).cpu(), torch.where(want == 0, want, torch.tensor(-10000.0)))


@pytest.mark.parametrize("sq,skv,kind", [(70, 333, "random"), (257, 512, "prefix"), (64, 97, "holes"), (33, 64, "one")])
def test_masked_attention_against_oracle(dev, sq, skv, kind):
  B, H = 2, 3
  q, k, v = O.normal_bf16((B, sq, H, 128), 0), O.normal_bf16((B, skv, H, 128), 1), O.normal_bf16((B, skv, H, 128), 2)
  rng = np.random.default_rng(5)
  keep = np.ones((B, skv), bool)
  if kind == "random":
    keep = rng.random((B, skv)) < 0.6
  elif kind == "prefix":  # padding masks: batch 0 keeps 300 keys, batch 1 keeps 77
    keep[0, 300:] = False
    keep[1, 77:] = False
  elif kind == "holes":  # whole 32-key tiles masked out, first tile included
    keep[0, :32] = False
    keep[1, 32:64] = False
    keep[1, 90:] = False
  else:  # a single kept key: out = that key's value row, lse = its logit
    keep[:] = False
    keep[0, 40] = True
    keep[1, 63] = True
  bias = ops.key_mask_bias(torch.from_numpy(keep).to(dev))
  out, lse = ops.flash_attention(to_dev_bf16(q, dev), to_dev_bf16(k, dev), to_dev_bf16(v, dev), return_lse=True, key_bias=bias)
  out, lse = to_np(out), to_np(lse)
  for b in range(B):
    ro, rl = O.attention(hsd(q[b:b + 1]), hsd(k[b:b + 1]), hsd(v[b:b + 1]), 128**-0.5, kv_mask=keep[b])
    mx, mean = err_stats(hsd(out[b:b + 1]), ro)
    lmx = float(np.abs(lse[b] - rl).max())
    print(f"mask {kind} Sq={sq} Skv={skv} batch {b}: out max-abs {mx:.3e} mean-abs {mean:.3e} rel-l2 {rel_l2(hsd(out[b:b+1]), ro):.3e} lse {lmx:.3e}", flush=True)
    assert mx <= MAX_ABS and mean <= MEAN_ABS and rel_l2(hsd(out[b:b + 1]), ro) <= REL_L2 and lmx <= LSE_ABS
  # the same mask with the softmax scale carried by q (scale = ln 2 for the kernel): the masked kernel keeps its
  # multiply, the result is the one of the plain call on these inputs
  qf = O.bf16_round((q * np.float32(ops.folded_q_mul(128))).astype(np.float32))
  out2, lse2 = ops.flash_attention(to_dev_bf16(qf, dev), to_dev_bf16(k, dev), to_dev_bf16(v, dev), scale=ops.FOLDED_SCALE,
                                   return_lse=True, key_bias=bias)
  for b in range(B):
    ro, rl = O.attention(hsd(qf[b:b + 1]), hsd(k[b:b + 1]), hsd(v[b:b + 1]), ops.FOLDED_SCALE, kv_mask=keep[b])
    mx, mean = err_stats(hsd(to_np(out2)[b:b + 1]), ro)
    assert mx <= MAX_ABS and mean <= MEAN_ABS and float(np.abs(to_np(lse2)[b] - rl).max()) <= LSE_ABS


def test_all_keys_masked_rows_return_zero_and_all_kept_equals_unmasked(dev):
  B, S, H = 2, 100, 2
  q, k, v = (to_dev_bf16(O.normal_bf16((B, S, H, 128), s), dev) for s in (0, 1, 2))
  keep = torch.ones((B, S), dtype=torch.bool, device=dev)
  keep[1] = False  # batch 1: nothing to attend to
  out, lse = ops.flash_attention(q, k, v, return_lse=True, key_bias=ops.key_mask_bias(keep))
  base, lse0 = ops.flash_attention(q, k, v, return_lse=True)
  # same arithmetic up to where the scale is applied (before instead of inside the exp2 argument): bf16 ulps
  assert torch.allclose(out[0].float(), base[0].float(), atol=2e-3, rtol=1e-2) and torch.allclose(lse[0], lse0[0], atol=1e-5)
  assert torch.count_nonzero(out[1]) == 0 and bool(torch.isneginf(lse[1]).all())


def test_reference_hand_fixture_and_dispatcher(dev):
  # tests/ltx2/test_attention_ltx2.py:38-76: two keys, the second masked -> every query returns v[0]
  H, D = 2, 128
  q = torch.randn(1, 5, H * D, device=dev).to(torch.bfloat16)
  k = torch.randn(1, 2, H * D, device=dev).to(torch.bfloat16)
  v = torch.randn(1, 2, H * D, device=dev).to(torch.bfloat16)
  op = attention_op.AttentionOp(attention_kernel="hip_flash", heads=H, dim_head=D, scale=D**-0.5)
  got = op.apply_attention(q, k, v, attention_mask=torch.tensor([[1, 0]], device=dev))
  assert got.shape == (1, 5, H * D)
  assert torch.equal(got, v[:, :1].expand(1, 5, H * D))
  # :91-116: everything masked -> zeros
  got = op.apply_attention(q, k, v, attention_mask=torch.tensor([[0, 0]], device=dev))
  assert torch.count_nonzero(got) == 0


@pytest.mark.parametrize("D", [128, 64, 80])
@pytest.mark.parametrize("skv,kind", [(384, "prefix257"), (4500, "prefix100"), (2200, "blocks"), (97, "last"), (333, "none"), (64, "all"), (2111, "holes")])
def test_masked_attention_visits_the_kept_tiles_only(dev, lib, D, skv, kind):
  """The registry entry's mask path (tile lists made on the device) against the same attention on the kept keys alone, forward
  and gradients: lists of one and several registers, tiles dropped in front, between and behind, none kept in one batch
  element.  f32 accumulation in another order only: bf16 bars of the unmasked kernels."""
  from maxdiffusion_amd import attention_op as A
  B, H, sq = 2, 2, 70
  gen = torch.Generator(device=dev).manual_seed(skv)
  keep = torch.zeros((B, skv), dtype=torch.bool, device=dev)
  if kind.startswith("prefix"):
    keep[:, :int(kind[6:])] = True
    keep[1, 40:] = False
  elif kind == "blocks":
    keep[0, 64:128] = keep[0, 1990:2100] = keep[1, 500:501] = True
  elif kind == "last":
    keep[:, skv - 1] = True
  elif kind == "all":
    keep[:] = True
  elif kind == "holes":
    keep[:] = torch.rand((B, skv), generator=gen, device=dev) < 0.05
    keep[0, 0] = keep[1, 7] = True
  else:
    keep[0, 3:200] = True  # nothing kept in element 1
  mk = lambda s: torch.randn((B, s, H * D), generator=gen, device=dev).to(torch.bfloat16).requires_grad_(True)
  q, k, v = mk(sq), mk(skv), mk(skv)
  g = torch.randn((B, sq, H * D), generator=gen, device=dev).to(torch.bfloat16)
  op = A.AttentionOp(attention_kernel="hip_flash", scale=D**-0.5, heads=H, dim_head=D, dtype=torch.bfloat16)
  out = op.apply_attention(q, k, v, attention_mask=keep)
  grads = torch.autograd.grad(out, (q, k, v), g)
  with torch.no_grad():
    assert torch.equal(op.apply_attention(q, k, v, attention_mask=keep), out)
  for b in range(B):
    idx = keep[b].nonzero()[:, 0]
    for t in (grads[1], grads[2]):
      assert not t[b][~keep[b]].any()
    if idx.numel() == 0:
      assert not out[b].any() and not grads[0][b].any()
      continue
    rq, rk, rv = (t.detach().float().requires_grad_(True) for t in (q[b], k[b, idx], v[b, idx]))
    hf = lambda t: t.view(-1, H, D).transpose(0, 1)
    ref = (torch.softmax((hf(rq) @ hf(rk).transpose(1, 2)) * D**-0.5, -1) @ hf(rv)).transpose(0, 1).reshape(sq, H * D)
    want = torch.autograd.grad(ref, (rq, rk, rv), g[b].float())
    for name, got, r in (("out", out[b], ref), ("dq", grads[0][b], want[0]), ("dk", grads[1][b, idx], want[1]), ("dv", grads[2][b, idx], want[2])):
      r = r.detach()
      if float(r.abs().max()) < 1e-5:  # a single key: the exact gradients of q and k are zero
        assert float(got.detach().float().abs().max()) <= 0.25, name
        continue
      rel = float((got.detach().float() - r).norm() / r.norm())
      assert rel <= 6e-3, (name, kind, rel)


def test_nan_in_a_key_bias_reaches_the_gradients(dev):
  """A NaN bias between excluded keys is not taken for another excluded key: the rows' outputs and the gradients of that key
  are NaN."""
  B, S, H, D = 1, 70, 2, 128
  gen = torch.Generator(device=dev).manual_seed(1)
  q, k, v, g = (torch.randn((B, S, H, D), generator=gen, device=dev).to(torch.bfloat16) for _ in range(4))
  bias = torch.full((B, 96), float("-inf"), device=dev)
  bias[0, 3] = float("nan")
  out, lse = ops.flash_attention(q, k, v, return_lse=True, key_bias=bias)
  dq, dk, dv = ops.flash_attention_backward(q, k, v, out, g, lse, key_bias=bias)
  for t in (out, lse, dq, dk[:, 3], dv[:, 3]):
    assert t.isnan().all()


@pytest.mark.parametrize("B,skv", [(1, 1), (3, 33), (2, 8191), (3, 8192), (2, 8193), (2, 24631), (1, 75600)])
@pytest.mark.parametrize("density", [1.0, 0.02, 0.0])
def test_key_tile_lists(dev, lib, B, skv, density):
  """The bias and the tile lists of a mask, against numpy: one slice of 8,192 keys and several, rows at any address."""
  rng = np.random.default_rng(skv)
  keep = rng.random((B, skv)) < density
  keep[B - 1, skv // 2:] = density > 0.5 and skv % 2 == 1  # an element that ends in dropped (or mixed and kept) tiles
  cols, ints = (skv + 31) // 32 * 32, lib.mdattn_host_key_tiles_ints
  ints.restype = ctypes.c_int64
  n = ints(B, skv)
  bias = torch.full((B, cols), 7.0, device=dev)
  tiles = torch.full((n,), -1, dtype=torch.int32, device=dev)
  kd = torch.from_numpy(keep).to(dev)
  rc = lib.mdattn_host_key_tiles(ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), ctypes.c_void_p(kd.data_ptr()), ctypes.c_void_p(bias.data_ptr()),
                                 ctypes.c_void_p(tiles.data_ptr()), B, skv, ctypes.c_int64(cols))
  assert rc == 0
  want = np.full((B, cols), -np.inf, np.float32)
  want[:, :skv][keep] = 0
  assert np.array_equal(bias.cpu().numpy(), want)
  got, at = tiles.cpu().numpy(), 0
  for ts in (32, 64):
    nt = (skv + ts - 1) // ts
    for b in range(B):
      kept = np.add.reduceat(keep[b].astype(int), np.arange(0, skv, ts))
      size = np.minimum(ts, skv - ts * np.arange(nt))
      entries = [2 * t + int(kept[t] < size[t]) for t in range(nt) if kept[t]]
      assert got[at] == len(entries) and list(got[at + 1:at + 1 + len(entries)]) == entries
      assert (got[at + 1 + len(entries):at + 1 + nt] == -1).all()
      at += 1 + nt
  assert at == n


@pytest.mark.parametrize("skv", [32, 33, 64, 65, 96, 97, 128, 129, 190])
def test_additive_bias_one_to_six_key_tiles(dev, skv):
  """Head dim 128: the first tile and the last are copies of the loop's body of their own; finite biases and an excluded key in
  every tile.  out and lse against float64."""
  H, sq = 3, 70
  q, k, v = O.normal_bf16((1, sq, H, 128), 0), O.normal_bf16((1, skv, H, 128), 1), O.normal_bf16((1, skv, H, 128), 2)
  bias = np.full((1, (skv + 31) // 32 * 32), -np.inf, np.float32)
  bias[0, :skv] = 3.0 * np.random.default_rng(skv).standard_normal(skv)
  bias[0, 5:skv:32] = -np.inf
  out, lse = ops.flash_attention(to_dev_bf16(q, dev), to_dev_bf16(k, dev), to_dev_bf16(v, dev), return_lse=True, key_bias=torch.from_numpy(bias).to(dev))
  logits = hsd(q).astype(np.float64) @ hsd(k).astype(np.float64).transpose(0, 2, 1) * 128**-0.5 + bias[0, :skv]
  m = logits.max(-1, keepdims=True)
  p = np.exp(logits - m)
  total = p.sum(-1, keepdims=True)
  assert rel_l2(hsd(to_np(out)), (p / total) @ hsd(v)) <= 6e-3  # bf16 roundings of the probabilities and of the output
  assert np.abs(to_np(lse)[0] - (m + np.log(total))[..., 0]).max() <= 1e-3
