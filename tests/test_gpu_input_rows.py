"""Inputs whose rows are not what the kernels read: misaligned starts and
strides of axes of one element."""
import pytest
import torch

from gpu_helpers import banner, seeded

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
