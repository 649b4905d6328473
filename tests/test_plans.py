"""How calls are launched, as the library plans it on the host: no GPU needed.  Each expectation is the faster of the forms timed on an
MI355X; the kernels' results under every plan are the GPU tests' business."""
import ctypes
import math
import random

import pytest

PIPELINED8, PIPELINED4, FLAT = 1, 2, 3


@pytest.mark.parametrize("H,sq,skv,plain,folded", [
    (12, 3193, 3195, PIPELINED8, PIPELINED8),  # 300 workgroups of 128 queries: 70 us, flat 79; folded 68 and 70
    (40, 900, 12795, PIPELINED8, PIPELINED8),
    (20, 1024, 4096, PIPELINED4, PIPELINED4),
    (12, 2680, 3000, PIPELINED4, PIPELINED4),
    (40, 2048, 4096, FLAT, FLAT),
    (40, 512, 512, FLAT, FLAT),
    (40, 75600, 512, FLAT, FLAT),
    (40, 75600, 75600, PIPELINED8, PIPELINED8),
])
def test_schedule_of_an_uncut_forward(lib, H, sq, skv, plain, folded):
  assert lib.mdattn_host_fwd_schedule(1, H, sq, skv, 128, 128**-0.5) == plain
  assert lib.mdattn_host_fwd_schedule(1, H, sq, skv, 128, math.log(2.0)) == folded
  assert lib.mdattn_host_fwd_schedule(1, H, sq, skv, 64, 0.125) == FLAT


class Pass(ctypes.Structure):
  _fields_ = [("waves", ctypes.c_int), ("pieces", ctypes.c_int), ("tiles", ctypes.c_int), ("floats", ctypes.c_int64)]


class Plan(ctypes.Structure):
  _fields_ = [("dq", Pass), ("dkv", Pass)]


def _plan(lib, B, H, sq, skv, D, bias, room=-1):
  p = Plan()
  n = lib.mdattn_host_bwd_plan_floats(B, H, sq, skv, D, bias, room, ctypes.addressof(p))
  as_tuple = lambda x: (x.waves, x.pieces, x.tiles, x.floats)
  return as_tuple(p.dq), as_tuple(p.dkv), n


# the first four came out differently with the space of their own plan as the limit
SHAPES = [(1, 4, 225, 11304, 128), (1, 4, 2324, 913, 128), (1, 2, 906, 14932, 80), (1, 12, 5887, 44, 128), (1, 12, 32760, 512, 128), (2, 32, 1337, 1337, 64),
          (1, 20, 18900, 18900, 128), (1, 1, 1, 1, 128)]


def _shapes():
  rng = random.Random(5)
  size = lambda: int(math.exp(rng.uniform(0, math.log(20000))))
  return SHAPES + [(rng.choice([1, 2]), rng.choice([1, 4, 5, 12, 24, 40]), size(), size(), rng.choice([128, 64, 80, 40])) for _ in range(2000)]


@pytest.mark.parametrize("bias", [0, 1])
def test_a_backward_is_launched_as_its_workspace_was_sized(lib, bias):
  for B, H, sq, skv, D in _shapes():
    dq, dkv, n = _plan(lib, B, H, sq, skv, D, bias)
    base = lib.mdattn_bwd_workspace_floats(B, H, sq)
    assert n == base + max(dq[3], 2 * dkv[3]) <= lib.mdattn_bwd_split_workspace_floats(B, H, sq, skv, D)
    assert _plan(lib, B, H, sq, skv, D, bias, n) == (dq, dkv, n)
    for room in (base, base + (n - base) // 2):  # less space: what fits, every tile walked once
      for (waves, pieces, tiles, floats), rows, other, tensors in zip(_plan(lib, B, H, sq, skv, D, bias, room)[:2], (sq, skv), (skv, sq), (1, 2)):
        nt = (other + 31) // 32
        assert waves in ((4, 8) if D > 64 else (4,)) and (pieces - 1) * tiles < nt <= pieces * tiles
        assert floats == (pieces * B * H * rows * D if pieces > 1 else 0) and tensors * floats <= room - base


@pytest.mark.parametrize("B,H,s,D", [(2, 4, 3572, 128), (1, 16, 1688, 40), (1, 16, 1688, 64)])
def test_a_masked_dq_pass_is_cut_where_its_tiles_are_dearer(lib, B, H, s, D):
  """Whole without a mask; under one 125 us whole and 93 in pieces, 45 and 33, 48 and 36."""
  assert _plan(lib, B, H, s, s, D, 0)[0][1] == 1
  assert _plan(lib, B, H, s, s, D, 1)[0][1] > 1


def test_backward_plan_refuses(lib):
  assert lib.mdattn_host_bwd_plan_floats(1, 4, 100, 100, 120, 0, -1, None) == 0
  assert lib.mdattn_host_bwd_plan_floats(1, 4, 100, 0, 128, 0, -1, None) == 0
  assert lib.mdattn_host_bwd_plan_floats(1, 4, 100, 100, 128, 0, lib.mdattn_bwd_workspace_floats(1, 4, 100) - 1, None) == 0


def test_a_plan_of_other_sizes_is_refused(lib):
  """Before anything is launched: a plan with too few pieces, pieces past the end or more space than the workspace has."""
  import torch

  from maxdiffusion_amd import _lib

  if torch.cuda.is_available():
    pytest.skip("the addresses below are nobody's: not where a kernel could be launched with them")
  B, H, sq, skv, D = 1, 12, 4096, 77, 128
  plan, L = Plan(), ctypes.c_int64
  n = lib.mdattn_host_bwd_plan_floats(B, H, sq, skv, D, 0, -1, ctypes.addressof(plan))
  assert plan.dkv.pieces > 1
  at, st = ctypes.c_void_p(4096), _lib.Strides(sq * H * D, H * D, D)

  def call(p, floats, keys=skv):
    return lib.mdattn_host_bwd_bf16(None, *[at] * 9, at, L(floats), B, H, sq, keys, D, *[ctypes.byref(st)] * 4, ctypes.c_float(0.1), None, L(0), None,
                                    ctypes.byref(p))

  assert call(plan, n - 1) == _lib.E_BADARG and call(plan, n, keys=skv + 32) == _lib.E_BADARG
  for field, value in (("pieces", plan.dkv.pieces - 1), ("pieces", plan.dkv.pieces + 1), ("tiles", plan.dkv.tiles - 1), ("waves", 2), ("floats", 0)):
    other = Plan.from_buffer_copy(plan)
    setattr(other.dkv, field, value)
    assert call(other, n) == _lib.E_BADARG, field
