"""The float32-MFMA forms that GM_SPLIT_PRODUCTS=0 selects, in one child process
(the library reads the switch once): bfloat16 node vectors' weight gradient,
which keeps the split kernels there, and the radial depthwise forward."""

import os
import subprocess
import sys
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu

TESTS = Path(__file__).resolve().parent

# The workspace is filled with NaN first: a partial matrix the kernels do not write must not be summed.  The bound is
# that of the split products (2^-22 of the sum of magnitudes) and a float32 chain's, its length times 2^-24.
WEIGHT_GRADIENT = """
import torch
from gm_attention_amd import _native
lib, cuda = _native.library(), torch.device("cuda:0")
for N, w, C in ((1, 17, 4), (33, 32, 260), (2048, 64, 544), (9000, 24, 132), (300, 33, 1028), (129, 16, 68)):
    print("weight gradient", N, w, C, flush=True)
    g = torch.Generator().manual_seed(N + w + C)
    v = torch.randn(N, w, generator=g).bfloat16().to(cuda)
    dmix = torch.randn(N, C, generator=g).to(cuda)
    partial = torch.full((lib.gm_node_mix_weight_partials(N, w, C),), float("nan"), device=cuda)
    dm = torch.full((w, C), float("nan"), device=cuda)
    status = lib.gm_node_mix_backward_weight_bf16(v.data_ptr(), w, dmix.data_ptr(), N, w, C, partial.data_ptr(),
                                                  dm.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert status == 0, lib.gm_last_error()
    want, size = v.double().t() @ dmix.double(), v.double().abs().t() @ dmix.double().abs()
    bound = size * (2.0 ** -22 + (6 * 128 + N // 4096 + 64) * 2.0 ** -24)
    assert bool(((dm.double() - want).abs() <= bound).all()), (N, w, C, float((dm.double() - want).abs().max()))
"""

RADIAL_FORWARD = """
import torch
import test_radial_forward_gpu as radial
for basis in (4, 8):
    for a0, orders in ((4, []), (0, [2]), (12, [1, 2, 2]), (20, [1] * 5 + [2] * 3), (32, [1, 2] * 8)):
        print("radial forward", basis, a0, orders, flush=True)
        radial.test_partial_and_mixed_groups_over_ragged_rows(a0, orders, basis, torch.device("cuda:0"))
"""


def test_the_forms_without_split_products(cuda):
    code = f"import sys; sys.path[:0] = {[str(TESTS), str(TESTS.parent), str(TESTS.parent / 'gm-attention_amd')]!r}\n"
    ran = subprocess.run([sys.executable, "-u", "-c", code + WEIGHT_GRADIENT + RADIAL_FORWARD], capture_output=True,
                         text=True, timeout=100, env={**os.environ, "GM_SPLIT_PRODUCTS": "0"})
    print(ran.stdout, flush=True)
    assert ran.returncode == 0, ran.stderr[-3000:]
