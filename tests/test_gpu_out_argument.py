"""``out=`` at head dims other than 64 and 128: the kernel writes a caller's
tensor directly only where that is the same as copying a finished result into
it, and everything ``copy_`` takes or refuses stays so."""
import pytest
import torch

from gpu_helpers import banner, seeded

pytestmark = pytest.mark.gpu

B, H, S = 2, 3, 150


@pytest.fixture(scope="module")
def sp():
  if not torch.cuda.is_available():
    pytest.skip("no GPU")
  from diffusers_tpu_amd.kernels import splash
  return splash


def _qkv(d):
  return [seeded((B, H, S, d), 670 + i) for i in range(3)]


@pytest.mark.parametrize("d", [72, 160])
@pytest.mark.parametrize("start", [1, 2, 3, 4])
def test_out_starts_anywhere(sp, d, start):
  banner(f"out at element {start}, dim {d}")
  q, k, v = _qkv(d)
  want = sp.attention(q, k, v)
  buf = torch.full((B, H, S, d + 4), 7.0, device="cuda", dtype=torch.bfloat16)
  out = buf[..., start:start + d] if start < 4 else buf[..., 4:]
  assert out.data_ptr() % 8 == (2 * start) % 8
  assert sp.attention(q, k, v, out=out) is out
  assert torch.equal(out, want)
  rest = torch.ones(d + 4, dtype=torch.bool)
  rest[start:start + d] = False
  assert (buf[..., rest.to("cuda")] == 7).all()


@pytest.mark.parametrize("d", [72, 160])
def test_out_as_copy_takes_it(sp, d):
  banner(f"out semantics, dim {d}")
  q, k, v = _qkv(d)
  want = sp.attention(q, k, v)
  # one element for many positions
  one = torch.zeros(B, H, 1, d, device="cuda", dtype=torch.bfloat16)
  with pytest.raises(RuntimeError):
    sp.attention(q, k, v, out=one.expand(-1, -1, S, -1))
  # an in-place write: the version counts, and a leaf that records refuses it
  out = torch.empty_like(q)
  version = out._version
  sp.attention(q, k, v, out=out)
  assert out._version > version and torch.equal(out, want)
  leaf = torch.zeros_like(q).requires_grad_()
  with pytest.raises(RuntimeError):
    sp.attention(q, k, v, out=leaf)
  with torch.no_grad():
    assert torch.equal(sp.attention(q, k, v, out=leaf), want)
  with torch.inference_mode():
    held = torch.empty_like(q)
    assert torch.equal(sp.attention(q, k, v, out=held), want)
  with pytest.raises(RuntimeError):
    sp.attention(q, k, v, out=held)


@pytest.mark.parametrize("d", [72, 160])
def test_out_over_an_input_through_another_storage(sp, d):
  """A view handed over by DLPack is a storage of its own over the same
  memory: rows must not be read after they are written."""
  banner(f"out over v, dim {d}")
  q, k, v = _qkv(d)
  want = sp.attention(q, k, v)
  buf = torch.zeros(v.numel() + 8 * d, device="cuda", dtype=torch.bfloat16)
  vv = buf[8 * d:].view(v.shape).copy_(v)
  out = torch.from_dlpack(buf[:v.numel()]).view(v.shape)
  assert sp._memory_overlaps(out, vv)
  sp.attention(q, k, vv, out=out)
  assert torch.equal(out, want)
  assert not sp._memory_overlaps(q, k)
