"""How calls are launched, as the library plans it on the host: no GPU needed.  Each expectation is the faster of the forms timed on an
MI355X; the kernels' results under every plan are the GPU tests' business."""
import math

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
