"""Rows whose scores lie far from zero, and keys that only some tiles see:
the kernels keep one reference per row, taken from the first tile they sweep,
so scores far below zero there, or a tile of masked keys (a channel that gives
-inf, or the type's lowest value) at the start of a key group's or a split
part's share must not reach the result."""
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


# (B, H, Sq, Skv, D): 4 x 2 and 2 x 4 key groups; split parts
MASKED = [(2, 22, 250, 1500, 128), (1, 8, 1000, 1024, 64), (1, 24, 300, 1500, 72),
          (1, 2, 300, 4096, 256), (1, 3, 200, 2500, 136),
          (1, 2, 300, 4096, 128), (1, 2, 300, 6000, 64), (1, 2, 300, 4096, 88)]


@pytest.mark.parametrize("low", [float("-inf"), torch.finfo(torch.bfloat16).min])
@pytest.mark.parametrize("case", MASKED, ids=[str(c) for c in MASKED])
def test_masked_tiles_after_the_first(dta, case, low):
  """All keys but tile 0 and a few of the last ones masked by a channel."""
  b, h, sq, skv, d = case
  from diffusers_tpu_amd.kernels.block_sizes import launch_shape
  banner(f"masked tiles {case} {low}")
  if torch.cuda.get_device_properties(0).multi_processor_count == 256:
    s = launch_shape(b, h, sq, skv, d)
    assert s.key_groups > 1 or s.split_parts > 1
  q, k, v = _inputs(b, h, sq, skv, d, 660)
  q[..., 0], k[..., 0] = 1.0, 0.0
  keep = np.r_[0:64, skv - 5:skv]
  want = A.attention_f64(to64(q[:1, :2]), to64(k[:1, :2, keep]),
                         to64(v[:1, :2, keep]))
  k[:, :, 64:skv - 5, 0] = low
  got = dta.attention(q, k, v)
  assert_attn_close(to64(got[:1, :2]), want, "masked")
  o, m, l = dta.residual_attention(q, k, v)
  assert_attn_close(to64((o / l)[:1, :2]), want, "residual")


@pytest.mark.parametrize("low", [float("-inf"), torch.finfo(torch.bfloat16).min])
@pytest.mark.parametrize("skv", [4000, 4096])
def test_masked_tiles_of_a_table(dta, skv, low):
  """Split parts of a tile table's sweep, whose first tile is any tile (the
  second query block lists only the last, partial one)."""
  from diffusers_tpu_amd.kernels import sparse_splash
  banner(f"masked tiles of a table, {skv} {low}")
  q, k, v = _inputs(1, 2, 500, skv, 128, 670)
  q[..., 0], k[..., 0] = 1.0, 0.0
  tiles = -(-skv // 64)
  rows = [[0] + list(range(2, tiles)), [tiles - 1]]
  k[:, :, 64:skv - 5, 0] = low
  got = sparse_splash.attention(q, k, v, block_q=256, block_kv=64, kv_table=rows)
  for lo, hi, keep in ((0, 256, np.r_[0:64, skv - 5:skv]),
                       (256, 500, np.r_[skv - 5:skv])):
    want = A.attention_f64(to64(q[:, :, lo:hi]), to64(k[:, :, keep]),
                           to64(v[:, :, keep]))
    assert_attn_close(to64(got[:, :, lo:hi]), want, f"rows {lo}:{hi}")
