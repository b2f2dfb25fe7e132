"""merge_residuals on GPU tensors (dt_merge_residuals): part counts at the
edges of the kernel's unrolled bounds, small rows, and calls that record or
transform torch operations, which keep going through torch."""
import pytest
import torch

from gpu_helpers import banner

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sp():
  if not torch.cuda.is_available():
    pytest.skip("no GPU")
  from diffusers_tpu_amd.kernels import splash
  return splash


def _parts(n, shape, seed=610):
  g = torch.Generator(device="cuda").manual_seed(seed)
  r = lambda *s: torch.randn(s, generator=g, device="cuda")
  return [(50 * r(*shape), 20 * r(*shape[:-1], 1),
           r(*shape[:-1], 1).abs() + 0.5) for _ in range(n)]


def _merge64(parts):
  ps = [[t.double() for t in p] for p in parts]
  big = torch.stack([p[1] for p in ps]).amax(0)
  o = sum(torch.exp2(p[1] - big) * p[0] for p in ps)
  return o / sum(torch.exp2(p[1] - big) * p[2] for p in ps)


@pytest.mark.parametrize("n", [1, 2, 3, 5, 8, 9, 16, 17])
@pytest.mark.parametrize("shape", [(1, 1, 1, 4), (2, 3, 65, 72),
                                   (1, 2, 130, 256)])
def test_merge_matches_64_bits(sp, n, shape):
  banner(f"merge {n} parts of {shape}")
  parts = _parts(n, shape)
  assert sp._merge_kernel_ok(parts) == (n <= 16)
  got = sp.merge_residuals(parts)
  want = _merge64(parts)
  # float32: exponents to |60| round at 2^-18, weights, sums and the division
  # to 2^-23 each, on terms that may cancel in the numerator
  ps = [[t.double() for t in p] for p in parts]
  big = torch.stack([p[1] for p in ps]).amax(0)
  mag = sum(torch.exp2(p[1] - big) * p[0].abs() for p in ps) / \
      sum(torch.exp2(p[1] - big) * p[2] for p in ps)
  assert got.dtype == torch.float32 and got.shape == want.shape
  assert ((got.double() - want).abs() <= 2.0**-16 * mag).all()


def test_merge_other_calls_go_through_torch(sp):
  banner("merge routes")
  parts = _parts(2, (1, 2, 9, 8))
  want = _merge64(parts).float()
  close = lambda t: torch.allclose(t, want, rtol=1e-4, atol=1e-4)
  # autograd
  leaf = [tuple(t.clone().requires_grad_() for t in p) for p in parts]
  out = sp.merge_residuals(leaf)
  out.sum().backward()
  assert close(out) and all(t.grad is not None for p in leaf for t in p)
  with torch.no_grad():
    assert sp._merge_kernel_ok(leaf) and close(sp.merge_residuals(leaf))
  # vmap and forward mode
  batched = [tuple(torch.stack([t, t]) for t in p) for p in parts]
  flat = [t for p in batched for t in p]
  f = lambda *ts: sp.merge_residuals([ts[:3], ts[3:]])
  assert close(torch.func.vmap(f)(*flat)[1])
  first = tuple(t for p in parts for t in p)
  o, tan = torch.func.jvp(f, first, tuple(torch.ones_like(t) for t in first))
  assert close(o) and tan.abs().max() > 0
  # strides, float64, a broadcast m
  tr = [tuple(t.transpose(1, 2).contiguous().transpose(1, 2) for t in p)
        for p in parts]
  assert not sp._merge_kernel_ok(tr) and close(sp.merge_residuals(tr))
  dbl = [tuple(t.double() for t in p) for p in parts]
  assert sp.merge_residuals(dbl).dtype == torch.float64
  assert sp.merge_residuals([tuple(t.cpu() for t in p) for p in parts]).is_cpu
  # the largest representable-apart m: the smaller part's weight is zero
  far = [(p[0], torch.full_like(p[1], v), p[2])
         for p, v in zip(parts, (-300.0, 100.0))]
  assert torch.equal(sp.merge_residuals(far), parts[1][0] / parts[1][2])


def test_merge_under_tracers(sp):
  """torch.jit.trace records the operations, and torch.fx passes proxies."""
  banner("merge: tracers")
  parts = _parts(2, (1, 2, 9, 8))
  other = _parts(2, (1, 2, 9, 8), seed=611)
  flat = lambda ps: tuple(t for p in ps for t in p)
  f = lambda *ts: sp.merge_residuals([ts[:3], ts[3:]])
  traced = torch.jit.trace(f, flat(parts))
  assert torch.allclose(traced(*flat(other)), _merge64(other).float(),
                        rtol=1e-4, atol=1e-4)

  def g(a, b):  # a, b: a part each, as one tensor of three planes
    return sp.merge_residuals([a, b])
  graph = torch.fx.symbolic_trace(g)
  ab = [torch.stack(torch.broadcast_tensors(*p)) for p in other]
  assert torch.allclose(graph(*ab), _merge64(other).float(), rtol=1e-4,
                        atol=1e-4)
