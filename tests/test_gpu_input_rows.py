"""Inputs whose rows are not what the kernels read: misaligned starts, strides
of axes of one element, key and value rows that overlap or repeat."""
import pytest
import torch

from gpu_helpers import assert_attn_close, banner, seeded, to64
from oracle import attention as A

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sp():
  if not torch.cuda.is_available():
    pytest.skip("no GPU")
  from diffusers_tpu_amd.kernels import splash
  return splash


def _misaligned(t):
  """The same values, contiguous, from an address off by 8 bytes."""
  flat = torch.empty(t.numel() + 4, device=t.device, dtype=t.dtype)
  out = flat[4:].view(t.shape)
  return out.copy_(t)


@pytest.mark.parametrize("d", [40, 72, 160, 256])
def test_misaligned_contiguous_inputs(sp, d):
  banner(f"misaligned inputs, dim {d}")
  q, k, v = (seeded((2, 3, 70, d), 680 + i) for i in range(3))
  want = sp.attention(q, k, v)
  got = sp.attention(*(_misaligned(t) for t in (q, k, v)))
  assert torch.equal(got, want)


@pytest.mark.parametrize("d", [40, 72, 160, 256])
def test_one_row_of_any_stride(sp, d):
  banner(f"one row, dim {d}")
  q, k, v = (seeded((2, 3, 1, d), 684 + i) for i in range(3))
  want = sp.attention(q, k, v)
  for stride in (0, 1, 3, 8):
    odd = [t.as_strided(t.shape, (*t.stride()[:2], stride, 1))
           for t in (q, k, v)]
    assert torch.equal(sp.attention(*odd), want), stride
  assert torch.equal(want, v)


@pytest.mark.parametrize("d", [64, 72, 128])
def test_key_rows_that_repeat_or_overlap(sp, d):
  """A row stride below the dim (0: one row for all positions): keys and
  values each, on every route (plain, converted query, residual, E4M3 keys,
  tile table, packed V), as the same rows written out."""
  from diffusers_tpu_amd.kernels import sparse_splash
  banner(f"overlapping rows, dim {d}")
  b, h, s = 2, 3, 150
  q, k, v = (seeded((b, h, s, d), 687 + i) for i in range(3))
  flat = seeded((b, h, 8 * s + d), 690)
  views = {"repeat": flat[:, :, :d].unsqueeze(2).expand(-1, -1, s, -1),
           "overlap": flat.unfold(2, d, 8)[:, :, :s]}
  routes = {
      "plain": sp.attention,
      "float32 query": lambda q, k, v: sp.attention(q.float(), k, v),
      "residual": lambda q, k, v: sp.residual_attention(q, k, v)[0],
      "E4M3": lambda q, k, v: sp.attention(q, k, v, qk_fp8=True),
      "table": lambda q, k, v: sparse_splash.attention(
          q, k, v, block_q=512, block_kv=64, kv_table=[[0, 2]]),
  }
  for name, t in views.items():
    assert t.stride(2) < d
    dense = t.contiguous()
    for route, fn in routes.items():
      for a, w in (((q, t, v), (q, dense, v)), ((q, k, t), (q, k, dense)),
                   ((q, t, t), (q, dense, dense))):
        assert torch.equal(fn(*a), fn(*w)), (name, route)
    assert_attn_close(to64(sp.attention(q, t, v)),
                      A.attention_f64(to64(q), to64(dense), to64(v)), name)
  # one key with a row stride of zero
  k1, v1 = (t[:, :, :1].as_strided((b, h, 1, d), (*t.stride()[:2], 0, 1))
            for t in (k, v))
  got = sp.attention(q, k1, v1)
  assert torch.equal(got, v1.expand_as(got))
