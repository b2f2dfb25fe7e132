"""Workgroup shapes of the dense bf16 kernel: few query blocks or few key tiles
run in 128- or 64-row workgroups, with the tiles dealt to key groups of one
workgroup.  Sizes at the edges of the row blocks (64, 128, 256 rows), of the
tiles (64 keys) and of the groups (fewer tiles than groups), against the
float64 oracle.  (Which shape each size runs in, and lengths that leave a
group without tiles: test_gpu_launch_shape.)"""
import numpy as np
import pytest
import torch

from gpu_helpers import assert_attn_close, banner, seeded, to64
from oracle import attention as A

pytestmark = pytest.mark.gpu

# (B, Hq, Hkv, Sq, Skv, lengths per sample or None, D)
CASES = [(b, hq, hkv, sq, skv, n, d)
         for d in (64, 128)
         for b, hq, hkv, sq, skv, n in [
             (1, 1, 1, 1, 1, None),            # one row, one key
             (1, 2, 2, 65, 64, None),          # one tile
             (2, 2, 1, 129, 300, (65, 0)),     # device lengths, one of them 0
             (1, 3, 3, 128, 1087, None),       # 17 tiles, the last of 63 keys
             (2, 4, 2, 255, 1300, (1281, 1)),  # 21 tiles against 1
             (1, 4, 4, 700, 2049, None),       # a last tile of one key
         ]]


@pytest.fixture(scope="module")
def dta():
  if not torch.cuda.is_available():
    pytest.skip("no GPU")
  import diffusers_tpu_amd
  return diffusers_tpu_amd


@pytest.mark.parametrize("case", CASES, ids=[str(c) for c in CASES])
def test_row_shapes_match_oracle(dta, case):
  b, hq, hkv, sq, skv, lens, d = case
  banner(f"row shapes {case}")
  q = seeded((b, hq, sq, d), 600)
  k = seeded((b, hkv, skv, d), 601)
  v = seeded((b, hkv, skv, d), 602)
  n = None if lens is None else torch.tensor(lens, device="cuda",
                                             dtype=torch.int32)
  out = dta.attention(q, k, v, kv_len=n)
  o, m, l = dta.residual_attention(q, k, v, kv_len=n)
  torch.cuda.synchronize()
  for i in range(b):
    length = skv if lens is None else lens[i]
    if length == 0:
      assert not out[i].any() and not o[i].any() and not l[i].any()
      continue
    q64, k64, v64 = (to64(t[i:i + 1]) for t in (q, k, v))
    want = A.attention_f64(q64, k64, v64, kv_len=length)
    assert_attn_close(to64(out[i:i + 1]), want, f"sample {i}")
    assert_attn_close(to64(o[i:i + 1]) / to64(l[i:i + 1]), want,
                      f"residual {i}")
    wo, wm, wl = A.residual_f64(q64, k64, v64, kv_len=length)
    # m + log2(l) does not depend on the reference m: the probabilities are
    # rounded to bf16 (2^-9 relative in l) and so is c*q (2^-9 of a score)
    lse = to64(m[i:i + 1]) + np.log2(to64(l[i:i + 1]))
    c = np.log2(np.e) / np.sqrt(float(d))
    kr = np.repeat(k64[:, :, :length], hq // hkv, axis=1)
    shift = 2.0**-9 * np.einsum("bhid,bhjd->bhij", np.abs(c * q64),
                                np.abs(kr)).max(-1)[..., None]
    assert (np.abs(lse - (wm + np.log2(wl))) <= shift + 2.0**-8).all()


@pytest.mark.parametrize("d", [64, 72, 128])
def test_queries_read_as_they_lie(dta, d):
  """128-row workgroups bring their q rows in by DMA: rows with gaps and the
  last, partial block; rows that overlap or repeat are read directly."""
  banner(f"q rows at dim {d}")
  h, sq, skv = 40, 700, 130
  k = seeded((1, h, skv, d), 641)
  v = seeded((1, h, skv, d), 642)
  wide = seeded((1, sq, h, d + 8), 643)
  flat = seeded((1, h, 8 * sq + d), 644)
  views = {
      "gaps": wide[..., :d].transpose(1, 2),
      "overlapping": flat.unfold(2, d, 8)[:, :, :sq],
      "one row": flat[:, :, :d].unsqueeze(2).expand(-1, -1, sq, -1),
  }
  wide[..., d:] = float("nan")
  for name, q in views.items():
    got = dta.attention(q, k, v)
    rows = np.r_[0:3, 125:131, 255:258, sq - 70:sq]
    want = A.attention_f64(to64(q[:, :, rows]), to64(k), to64(v))
    assert_attn_close(to64(got[:, :, rows]), want, name)
