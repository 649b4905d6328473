"""The work a user of this framework has it do: attention blocks of the DiT models it serves, through the public entry
points (`AttentionOp.apply_attention`, the `hip_norm_rope*` hooks, the ring step), in inference and in training.

A case is one call of one block on one batch that is already on the GPU.  `path` names the kind of block:

  wan_self    q | k RMSNorm over all heads + rotation, self-attention (`fused`: over one q|k|v projection output with biases)
  wan_cross   norm only, the image tokens against a few hundred text keys; with `image_keys`, also against the image
              encoder's tokens, whose padding is masked, and the two results added
  flux        per-head RMSNorm with text / image weights + rotation, joint attention
  ltx2        full-row RMSNorm of f32 projections with f32 weights, per-head rotary tables, self-attention
  fp8         wan_self with the fp8 kernel
  ring        one rank's shard of context parallelism: its queries against the key / value chunks that pass by
  plain       the registry entry alone: any head dim up to 128, with or without a padding mask

`train` adds the backward pass: the gradients of every input and norm weight are returned with the output.  Values are
what projections of a normalised residual stream give: N(0, 1) in the compute type, norm weights around 1.
"""
import math

import torch

from maxdiffusion_amd import attention_op as A
from maxdiffusion_amd import ops

DEV = "cuda"


def listed():
  return [
      # the smallest call in the repository's own smoke run (4 heads, a 3 x 6 x 7 latent): what a call costs in latency
      dict(name="wan_tiny", path="wan_self", train=False, fused=False, batch=1, heads=4, frames=3, rows=6, cols=7),
      # Wan-1.3B (12 heads) on a short clip, 4,680 tokens: an ordinary interactive generation step
      dict(name="wan1.3b", path="wan_self", train=False, fused=False, batch=1, heads=12, frames=3, rows=30, cols=52),
      # Wan-14B (40 heads) on an 81-frame 720p clip, 75,600 tokens: the headline workload, the largest single call
      dict(name="wan14b", path="wan_self", train=False, fused=False, batch=1, heads=40, frames=21, rows=45, cols=80),
      # the cross-attention that follows it in every image-to-video block: 512 text keys, and 257 image tokens padded to 384
      dict(name="wan14b_i2v_cross", path="wan_cross", train=False, batch=1, heads=40, tokens=75600, keys=512, image_keys=257),
      # training one rank of 8 at that size (half of the heads, a quarter of the tokens), one q|k|v projection with biases
      dict(name="wan14b_shard_train", path="wan_self", train=True, fused=True, batch=1, heads=20, frames=21, rows=18, cols=50),
      # fine-tuning Wan-1.3B at 480p: its cross-attention, forward and backward
      dict(name="wan1.3b_cross_train", path="wan_cross", train=True, batch=1, heads=12, tokens=32760, keys=512, image_keys=0),
      # Flux-dev at 1024 x 1024 (24 heads, 512 text + 4,096 image tokens), a training step
      dict(name="flux_train", path="flux", train=True, batch=1, heads=24, text=512, rows=64, cols=64),
      # LTX-2's video stream (32 heads of 128): f32 projections, tables of the size of the tensor
      dict(name="ltx2_video", path="ltx2", train=False, rope="interleaved", batch=1, heads=32, head_dim=128, tokens=13376),
      # training on LTX-2's audio stream (32 heads of 64), two short ragged clips, the split rotation
      dict(name="ltx2_audio_train", path="ltx2", train=True, rope="split", batch=2, heads=32, head_dim=64, tokens=1337),
      # Wan-14B through the fp8 entry on a 480p clip
      dict(name="wan14b_fp8", path="fp8", batch=1, heads=40, frames=21, rows=30, cols=52),
      # one rank of an 8-way ring over the headline sequence: 9,450 queries, eight chunks of 9,450 keys
      dict(name="wan14b_ring", path="ring", batch=1, heads=40, tokens=9450, chunks=8),
      # an image encoder: 257 tokens, 16 heads of 80, a batch of frames
      dict(name="encoder_d80", path="plain", train=False, batch=16, heads=16, head_dim=80, tokens=257, keys=257, kept=257),
  ]


def _log(rng, lo, hi):
  return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
  """One more case: any of the paths, sizes spread over the logarithm of its range, cut where it would cost more than half
  of the largest listed case."""
  while True:
    path = rng.choice(["wan_self", "wan_self", "wan_cross", "wan_cross", "flux", "ltx2", "ltx2", "fp8", "ring", "plain", "plain"])
    c = dict(path=path, batch=rng.choice([1, 1, 1, 2, 4]))
    if path in ("wan_self", "fp8"):
      c.update(heads=rng.choice([4, 5, 12, 20, 40]), frames=rng.choice([1, 3, 9, 13, 21]), rows=_log(rng, 6, 45), cols=_log(rng, 7, 80))
      if path == "wan_self":
        c.update(train=rng.random() < 0.5, fused=rng.random() < 0.5)
    elif path == "wan_cross":
      c.update(train=rng.random() < 0.5, heads=rng.choice([4, 5, 12, 20, 40]), tokens=_log(rng, 100, 75600), keys=rng.choice([77, 256, 512, 512]),
               image_keys=rng.choice([0, 0, 257, 577]))
    elif path == "flux":
      c.update(train=rng.random() < 0.5, heads=24, text=rng.choice([128, 256, 512]), rows=_log(rng, 8, 96), cols=_log(rng, 8, 96))
    elif path == "ltx2":
      c.update(train=rng.random() < 0.5, rope=rng.choice(["interleaved", "split"]), heads=32, head_dim=rng.choice([64, 128]), tokens=_log(rng, 126, 13376))
    elif path == "ring":
      c.update(heads=rng.choice([5, 12, 40]), tokens=_log(rng, 300, 9450), chunks=rng.choice([2, 4, 8]))
    else:
      c.update(train=rng.random() < 0.3, heads=rng.choice([4, 10, 16, 20]), head_dim=rng.choice([40, 64, 64, 80, 96, 128]), tokens=_log(rng, 64, 8192))
      c["keys"] = c["tokens"] if rng.random() < 0.6 else _log(rng, 77, 2048)
      c["kept"] = c["keys"] if rng.random() < 0.5 else max(1, int(c["keys"] * rng.uniform(0.2, 0.95)))
    w = work(c)
    if w["flops"] <= 5e13 and w["bytes"] <= 3e10:
      return c


# ------------------------------------------------------------------------------------------------ inputs
def _tokens(c):
  if c["path"] in ("wan_self", "fp8"):
    return c["frames"] * c["rows"] * c["cols"]
  if c["path"] == "flux":
    return c["text"] + c["rows"] * c["cols"]
  return c["tokens"]


def _rope(axes, dims):
  """complex64 [S, sum(dims)/2]: one rotation per position and channel pair, each axis with its share of the channels."""
  ang = []
  for pos, d in zip(axes, dims):
    freq = 10000.0 ** (-torch.arange(0, d, 2, device=DEV, dtype=torch.float64) / d)
    ang.append(pos.reshape(-1, 1).double() * freq)
  a = torch.cat(ang, dim=1)
  return torch.polar(torch.ones_like(a), a).to(torch.complex64)


def _grid(f, r, w):
  return torch.meshgrid(*(torch.arange(n, device=DEV) for n in (f, r, w)), indexing="ij")


class _Maker:
  def __init__(self, seed, train):
    self.gen = torch.Generator(device=DEV).manual_seed(seed)
    self.train = train

  def normal(self, *shape, dtype=torch.bfloat16, std=1.0, leaf=True):
    x = torch.randn(shape, generator=self.gen, device=DEV, dtype=torch.float32).mul_(std).to(dtype)
    return x.requires_grad_(self.train and leaf)

  def weight(self, n, dtype=torch.bfloat16):
    x = (1 + 0.1 * torch.randn(n, generator=self.gen, device=DEV, dtype=torch.float32)).to(dtype)
    return x.requires_grad_(self.train)


def _op(kernel, heads, d, scale):
  return A.AttentionOp(attention_kernel=kernel, scale=scale, heads=heads, dim_head=d, dtype=torch.bfloat16)


def prepare(case, seed):
  c = dict(case)
  B, H, path = c["batch"], c["heads"], c["path"]
  D = c.get("head_dim", 128)
  S, N = _tokens(c), H * D
  mk = _Maker(seed, c.get("train", False))
  s = dict(case=c, folded=ops.folded_q_mul(D))
  s["op"] = _op("hip_flash_fp8" if path == "fp8" else "hip_flash", H, D, D**-0.5 if path in ("plain", "fp8") else ops.FOLDED_SCALE)
  if path in ("wan_self", "fp8"):
    if c.get("fused"):
      s.update(qkv=mk.normal(B, S, 3 * N), bias=mk.normal(3 * N, std=0.2))
    else:
      s.update(q=mk.normal(B, S, N), k=mk.normal(B, S, N), v=mk.normal(B, S, N))
    # the complex table [1, 1, S, D/2] as the model's rotary embedding returns it
    s.update(wq=mk.weight(N), wk=mk.weight(N), freqs=_rope(_grid(c["frames"], c["rows"], c["cols"]), (44, 42, 42))[None, None])
  elif path == "wan_cross":
    s.update(q=mk.normal(B, S, N), k=mk.normal(B, c["keys"], N), v=mk.normal(B, c["keys"], N), wq=mk.weight(N), wk=mk.weight(N))
    if c["image_keys"]:
      padded = (c["image_keys"] + 127) // 128 * 128
      keep = torch.zeros((B, padded), dtype=torch.bool, device=DEV)
      keep[:, :c["image_keys"]] = True
      s.update(ki=mk.normal(B, padded, N), vi=mk.normal(B, padded, N), wki=mk.weight(N), keep=keep, op_img=_op("hip_flash", H, D, D**-0.5))
  elif path == "flux":
    s.update(q=mk.normal(B, S, H, D), k=mk.normal(B, S, H, D), v=mk.normal(B, S, H, D))
    s.update({n: mk.weight(D) for n in ("wq", "wk", "wq_txt", "wk_txt")})
    ids = [torch.cat([torch.zeros(c["text"], device=DEV, dtype=torch.int64), x.reshape(-1)]) for x in _grid(1, c["rows"], c["cols"])]
    f = _rope(ids, (16, 56, 56))
    s["freqs"] = tuple(t.repeat_interleave(2, dim=1).contiguous() for t in (f.real, f.imag))  # each angle for both of its pair
  elif path == "ltx2":
    f32 = torch.float32
    s.update(q=mk.normal(B, S, N, dtype=f32), k=mk.normal(B, S, N, dtype=f32), v=mk.normal(B, S, N), wq=mk.weight(N, f32), wk=mk.weight(N, f32))
    ang = torch.rand((B, S, N // 2), generator=mk.gen, device=DEV) * (2 * math.pi)
    if c["rope"] == "interleaved":
      ang = ang.repeat_interleave(2, dim=2)
    else:
      ang = ang.view(B, S, H, D // 2).permute(0, 2, 1, 3).contiguous()
    s["freqs"] = (torch.cos(ang), torch.sin(ang))
  elif path == "ring":
    T = S * c["chunks"]
    s.update(q=mk.normal(B, S, H, D, std=ops.folded_q_mul(D)), k=mk.normal(B, T, H, D), v=mk.normal(B, T, H, D))
  else:
    s.update(q=mk.normal(B, S, N), k=mk.normal(B, c["keys"], N), v=mk.normal(B, c["keys"], N), keep=None)
    if c["kept"] < c["keys"]:
      s["keep"] = torch.zeros((B, c["keys"]), dtype=torch.bool, device=DEV)
      s["keep"][:, :c["kept"]] = True
  if c.get("train"):
    s["dout"] = mk.normal(B, S, N, leaf=False)
  return s


# ------------------------------------------------------------------------------------------------ one pass
def _rank3(x):
  return x.reshape(x.shape[0], x.shape[1], -1)


def _forward(s):
  c, op, H = s["case"], s["op"], s["case"]["heads"]
  path = c["path"]
  if path == "wan_self" and c["fused"]:
    q, k, v = A.hip_norm_rope_qkv(s["qkv"], s["wq"], s["wk"], s["freqs"], H, bias=s["bias"], q_mul=s["folded"])
    return op.apply_attention(_rank3(q), _rank3(k), _rank3(v))
  if path == "wan_self":
    q, k = A.hip_norm_rope(s["q"], s["k"], s["wq"], s["wk"], s["freqs"], H, q_mul=s["folded"])
    return op.apply_attention(_rank3(q), _rank3(k), s["v"])
  if path == "fp8":  # the entry quantises q with the softmax scale itself
    q, k = A.hip_norm_rope(s["q"], s["k"], s["wq"], s["wk"], s["freqs"], H)
    return op.apply_attention(_rank3(q), _rank3(k), s["v"])
  if path == "wan_cross":
    q, _ = A.hip_norm_rope(s["q"], None, s["wq"], None, None, H, q_mul=s["folded"])
    k, _ = A.hip_norm_rope(s["k"], None, s["wk"], None, None, H)
    out = op.apply_attention(_rank3(q), _rank3(k), s["v"])
    if c["image_keys"]:
      ki, _ = A.hip_norm_rope(s["ki"], None, s["wki"], None, None, H)
      out = out + s["op_img"].apply_attention(s["q"], _rank3(ki), s["vi"], attention_mask=s["keep"])
    return out
  if path == "flux":
    q, k = A.hip_norm_rope(s["q"], s["k"], s["wq"], s["wk"], s["freqs"], H, per_head=True, wq_txt=s["wq_txt"], wk_txt=s["wk_txt"],
                           n_txt=c["text"], q_mul=s["folded"])
    return op.apply_attention(_rank3(q), _rank3(k), _rank3(s["v"]))
  if path == "ltx2":
    q, k = A.hip_norm_rope_ltx2(s["q"], s["k"], s["wq"], s["wk"], H, rotary_emb=s["freqs"], rope_type=c["rope"], q_mul=s["folded"])
    return op.apply_attention(_rank3(q), _rank3(k), s["v"])
  return op.apply_attention(s["q"], s["k"], s["v"], attention_mask=s["keep"])


_LEAVES = ("qkv", "bias", "q", "k", "v", "ki", "vi", "wq", "wk", "wki", "wq_txt", "wk_txt")


def run(state):
  s, c = state, state["case"]
  if c["path"] == "ring":
    B, S, H, D = s["q"].shape
    o_run, lse_run = ops.new_merge_state(B, S, H, D, s["q"].device)
    for i in range(c["chunks"]):
      rows = slice(i * S, (i + 1) * S)
      ops.flash_attention_merge(s["q"], s["k"][:, rows], s["v"][:, rows], o_run, lse_run, scale=ops.FOLDED_SCALE)
    return ops.finalize(o_run), lse_run
  if not c.get("train"):
    with torch.no_grad():
      return _forward(s)
  out = _forward(s)
  leaves = [s[n] for n in _LEAVES if n in s]
  return out.detach(), torch.autograd.grad(out, leaves, s["dout"])


# ------------------------------------------------------------------------------------------------ what it cannot do without
def work(case):
  c, path = case, case["path"]
  B, H, D, S = c["batch"], c["heads"], c.get("head_dim", 128), _tokens(case)
  N = H * D
  train = c.get("train", False)
  keys = c["keys"] if path == "wan_cross" else c["kept"] if path == "plain" else S * c.get("chunks", 1)
  keys += c.get("image_keys", 0)
  # two matrix products forward; five more backward
  flops = 4.0 * B * H * S * keys * D * (3.5 if train else 1.0)
  q_bytes, k_bytes = (4, 4) if path == "ltx2" else (2, 2)
  nbytes = B * S * N * (q_bytes + 2.0) + B * keys * N * (k_bytes + 2.0)  # q read and out written; the keys and values that take part
  if train:
    nbytes += B * S * N * (q_bytes + 2.0) + B * keys * N * (k_bytes + 2.0)  # dout read, dq written; dk, dv written
  if path in ("wan_self", "fp8", "flux"):
    nbytes += S * D * 4.0 * (2 if path == "flux" else 1)  # the rotary table
  elif path == "ltx2":
    nbytes += B * S * N * (8.0 if c["rope"] == "interleaved" else 4.0)
  elif path == "ring":
    nbytes += B * H * S * 4.0
  return {"bytes": nbytes, "flops": flops}


def tolerance(case):
  # against the same block in 64 bits the bf16 paths are 2.5e-3 to 4.5e-3 off in every output and gradient; with the
  # value bias of the fused projection (the outputs' common part, which leaves nothing in the gradients of q and k) up to
  # 6e-3.  fp8: the rounding of the probabilities to e4m3 alone moves an output by 3e-2.
  if case["path"] == "fp8":
    return {"rel": 3e-2}
  return {"rel": 2.5e-2 if case.get("fused") and case.get("train") else 1.6e-2 if case.get("train") else 1.2e-2}
