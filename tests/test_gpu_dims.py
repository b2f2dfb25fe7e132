"""Head dims that are no kernel width (dt_flash_fwd_anydim): every count of QK
steps and output blocks, row blocks and the tail split, views whose rows are
not dense, outputs that share memory with an input."""
import numpy as np
import pytest
import torch

from gpu_helpers import assert_attn_close, banner, seeded, to64
from oracle import attention as A

pytestmark = pytest.mark.gpu

SHAPES = [
    # (B, Hq, Hkv, Sq, Skv, kv_len)
    (1, 1, 1, 1, 1, None),
    (2, 4, 2, 129, 200, 131),
    (1, 2, 2, 300, 4096, None),     # split parts (key groups up to 64)
    (1, 3, 3, 4200, 130, None),     # many row blocks, a short sweep
]


@pytest.fixture(scope="module")
def sp():
  if not torch.cuda.is_available():
    pytest.skip("no GPU")
  from diffusers_tpu_amd.kernels import splash
  return splash


def _want(q, k, v, n=None, rows=None):
  q64 = to64(q if rows is None else q[:, :, rows])
  return A.attention_f64(q64, to64(k), to64(v), kv_len=n)


@pytest.mark.parametrize("d", [8, 32, 40, 48, 56, 72, 80, 88, 96, 104, 112,
                               120, 136, 160, 168, 192, 224, 248, 256])
@pytest.mark.parametrize("shape", SHAPES, ids=[str(s) for s in SHAPES])
def test_dim_matches_oracle(sp, d, shape):
  b, hq, hkv, sq, skv, n = shape
  banner(f"dim {d} {shape}")
  q = seeded((b, hq, sq, d), 620)
  k = seeded((b, hkv, skv, d), 621)
  v = seeded((b, hkv, skv, d), 622)
  out = sp.attention(q, k, v, kv_len=n)
  o, m, l = sp.residual_attention(q, k, v, kv_len=n)
  torch.cuda.synchronize()
  assert out.shape == q.shape == o.shape and out.is_contiguous()
  rows = np.unique(np.r_[0:min(sq, 300), max(0, sq - 70):sq])
  want = _want(q, k, v, n, rows)
  assert_attn_close(to64(out[:, :, rows]), want, f"dim {d}")
  assert_attn_close(to64((o / l)[:, :, rows]), want, f"residual dim {d}")
  assert torch.isfinite(o).all()


@pytest.mark.parametrize("d", [40, 72, 112, 152])
def test_views_and_outputs(sp, d):
  banner(f"dim {d}: views")
  b, h, s = 2, 3, 150
  base = [seeded((b, s, h, d + 8), 623 + i) for i in range(3)]
  q, k, v = (t[..., :d].transpose(1, 2) for t in base)  # row gaps, BSHD
  want = _want(q, k, v)
  assert_attn_close(to64(sp.attention(q, k, v)), want, "BSHD rows with gaps")
  # NaN between the rows and past the key length stays out
  for t in base:
    t[..., d:] = float("nan")
  base[1][:, 100:] = float("nan")
  base[2][:, 100:] = float("nan")
  got = sp.attention(q, k, v, kv_len=100)
  assert_attn_close(to64(got), _want(q, k[:, :, :100], v[:, :, :100]),
                    "NaN outside")
  # one key row for all positions; overlapping rows
  q, k, v = (seeded((b, h, s, d), 626 + i) for i in range(3))
  ke = k[:, :, :1].expand(-1, -1, s, -1)
  assert_attn_close(to64(sp.attention(q, ke, v)), _want(q, ke, v), "expanded")
  flat = seeded((b, h, 8 * s + d), 629)
  kw = flat.unfold(2, d, 8)[:, :, :s]
  assert kw.stride(2) == 8
  assert_attn_close(to64(sp.attention(q, kw, v)), _want(q, kw, v), "windows")
  # out: strided rows of 8-byte alignment, and one that shares memory with v
  want = _want(q, k, v)
  wide = torch.zeros(b, h, s, d + 4, device="cuda", dtype=torch.bfloat16)
  out = wide[..., :d]
  assert sp.attention(q, k, v, out=out) is out
  assert_attn_close(to64(out), want, "8-byte rows")
  assert not wide[..., d:].any()
  assert sp.attention(q, k, v, out=v) is v
  assert_attn_close(to64(v), want, "out is v")


@pytest.mark.parametrize("d", [88, 200, 256])
def test_fixed_m_and_device_lengths(sp, d):
  banner(f"dim {d}: fixed-m, device lengths")
  q, k, v = (seeded((2, 4, 140, d), 630 + i) for i in range(3))
  k = (k.float() - k.float().mean(dim=2, keepdim=True)).to(torch.bfloat16)
  got = sp.attention(q, k, v, use_fixed_m=True)
  assert_attn_close(to64(got), _want(q, k, v), "fixed-m")
  n = torch.tensor([140, 0], device="cuda", dtype=torch.int32)
  got = sp.attention(q, k, v, kv_len=n)
  assert_attn_close(to64(got[:1]), _want(q[:1], k[:1], v[:1]), "length")
  assert not got[1].any()
  o, m, l = sp.residual_attention(q, k, v, kv_len=n)
  assert not o[1].any() and not m[1].any() and not l[1].any()


@pytest.mark.parametrize("d", [136, 256])
def test_wide_dims_split_only_long_sweeps(sp, d):
  """Half a round of workgroups is split over 4096 keys and not over 424,
  where the merge would cost more than the idle CUs."""
  banner(f"wide split plan d={d}")
  assert sp._split_bytes(2, 16, 424, 424, 424, d, 0) == 0
  assert sp._split_bytes(2, 16, 424, 4096, 4096, d, 0) > 0
