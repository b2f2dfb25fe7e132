"""Rows whose scores lie far from zero.  The kernels keep one reference per
row, set on the first tile they sweep."""
import numpy as np
import pytest
import torch

from gpu_helpers import assert_attn_close, banner, seeded, to64
from oracle import attention as A

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dta():
  if not torch.cuda.is_available():
    pytest.skip("no GPU")
  import diffusers_tpu_amd
  return diffusers_tpu_amd


def _inputs(b, h, sq, skv, d, seed):
  return (seeded((b, h, sq, d), seed), seeded((b, h, skv, d), seed + 1),
          seeded((b, h, skv, d), seed + 2))


# (B, H, Sq, Skv): key groups or 128-row blocks, split parts, whole sweeps
SHAPES = [(1, 2, 300, 300), (1, 4, 2600, 4096), (1, 300, 200, 200)]


@pytest.mark.parametrize("d", [64, 72, 128, 256])
@pytest.mark.parametrize("shape", SHAPES, ids=[str(s) for s in SHAPES])
def test_scores_far_below_zero(dta, d, shape):
  """Every score of a row near -512: the softmax is the one without the
  offset (channel 0 adds 16 * -32 sqrt(d) to q.k exactly in bf16)."""
  banner(f"low scores d={d} {shape}")
  q, k, v = _inputs(*shape, d, 650)
  off = 32.0 * 2.0**np.ceil(np.log2(np.sqrt(d)))
  q[..., 0], k[..., 0] = 16.0, 0.0
  h = sorted({0, shape[1] - 1})
  rows = np.r_[0:3, shape[2] - 3:shape[2]]
  # (bf16 of c*q takes the offset off by one factor for all keys of a row)
  want = A.attention_f64(to64(q[:, h][:, :, rows]), to64(k[:, h]),
                         to64(v[:, h]))
  k[..., 0] = -off
  got = dta.attention(q, k, v)
  assert_attn_close(to64(got[:, h][:, :, rows]), want, "offset")
  o, m, l = dta.residual_attention(q, k, v)
  assert_attn_close(to64((o / l)[:, h][:, :, rows]), want, "residual")

