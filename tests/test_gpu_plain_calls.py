"""The short host path of a plain attention call against the general path:
the same bits over layouts, lengths, residual outputs and workspaces, and the
same refusals.  Calls that the short path leaves to the general one are among
them.  Also the kernels of other head dims and of the residual merge under
HIP graph capture."""
import pytest
import torch

from gpu_helpers import banner, seeded
from test_gpu_graph import _replay_check

pytestmark = pytest.mark.gpu

B, H, S = 2, 4, 300


@pytest.fixture(scope="module")
def splash():
  if not torch.cuda.is_available():
    pytest.skip("no GPU")
  from diffusers_tpu_amd.kernels import splash
  return splash


def layouts(d):
  """(name, taken by the short path, q, k, v)"""
  q, k, v = (seeded((B, H, S, d), 900 + i) for i in range(3))
  yield "bhsd", True, q, k, v
  yield ("bshd", True) + tuple(t.transpose(1, 2).contiguous().transpose(1, 2)
                               for t in (q, k, v))
  fused = torch.cat([q, k, v], dim=-1)
  yield ("fused", True) + tuple(fused[..., i * d:(i + 1) * d] for i in range(3))
  yield "gqa", True, q, k[:, :2], v[:, :2]
  odd = torch.cat([k, v[..., :4]], dim=-1)[..., 4:]   # 8 bytes off, odd strides
  yield "misaligned", False, q, odd, v
  yield "float32", False, q.float(), k, v
  yield "columns", False, q, k, v.transpose(2, 3).contiguous().transpose(2, 3)


def lengths():
  dev = lambda *n: torch.tensor(n, device="cuda", dtype=torch.int32)
  return (("none", True, None), ("int", True, 65), ("device", True, dev(129)),
          ("per sample", True, dev(300, 0)), ("list", False, [257, 1]),
          ("int64", False, dev(129).long()))


@pytest.mark.parametrize("d", [64, 128])
def test_short_path_gives_the_general_paths_bits(splash, monkeypatch, d):
  banner(f"plain calls d={d}")
  short = splash._launch_plain

  def run(*args, **kw):
    try:
      return splash._launch(*args, **kw)
    except (ValueError, TypeError, NotImplementedError) as e:
      return type(e), str(e)

  for lname, fits, q, k, v in layouts(d):
    for nname, lfits, n in lengths():
      for residual in (False, True):
        for ws in (None, splash.AttentionWorkspace()):
          what = (lname, nname, residual, ws is not None)
          taken = short(q, k, v, None, n, residual, ws) is not None
          assert taken == (fits and lfits), what
          kw = dict(residual=residual, workspace=ws)
          got = run(q, k, v, None, n, **kw)
          with monkeypatch.context() as m:
            m.setattr(splash, "_launch_plain", lambda *a: None)
            want = run(q, k, v, None, n, **kw)
          if not residual:
            got, want = (got,), (want,)
          for x, y in zip(got, want):
            if isinstance(x, torch.Tensor):
              assert torch.equal(x, y) and x.stride() == y.stride(), what
            else:
              assert x == y, what


def test_short_path_leaves_wrong_calls_to_the_general_one(splash):
  banner("plain calls: refusals")
  q, k, v = (seeded((B, H, S, 64), 910 + i) for i in range(3))
  for exc, args, kw in (
      (ValueError, (q, k, v[:, :, :-1]), {}),
      (ValueError, (q[:1], k, v), {}),
      (ValueError, (q, k[:, :3], v[:, :3]), {}),
      (ValueError, (q, k, v), dict(kv_len=S + 1)),
      (ValueError, (q, k, v), dict(scale=-1.0)),
      (ValueError, (q[0], k[0], v[0]), {}),
      (ValueError, (q, k.cpu(), v.cpu()), {}),
      (TypeError, (q, k, v), dict(workspace=object()))):
    with pytest.raises(exc):
      splash.attention(*args, **kw)


@pytest.mark.parametrize("d", [72, 160])
def test_other_head_dims_and_merge_replay_in_a_graph(splash, d):
  banner(f"graph: residual halves at head dim {d}, merged")
  q, k, v = (seeded((1, 6, 700, d), 920 + i) for i in range(3))
  out = torch.empty((1, 6, 700, d), device="cuda", dtype=torch.float32)
  ws = splash.AttentionWorkspace()

  def step():
    parts = [splash.residual_attention(q, k[:, :, a:b], v[:, :, a:b],
                                       workspace=ws)
             for a, b in ((0, 333), (333, 700))]
    out.copy_(splash.merge_residuals(parts))

  _replay_check(step, out)
