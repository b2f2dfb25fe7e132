"""Every workgroup shape of the dense bf16 kernel at every kernel width, the
shape that runs asserted: against the float64 oracle, with per-sample lengths
that end inside a tile and that leave key groups and split parts without tiles,
and packed V against row-major V bit for bit."""
import numpy as np
import pytest
import torch

from gpu_helpers import assert_attn_close, banner, seeded, to64
from oracle import attention as A

pytestmark = pytest.mark.gpu

# (rows, key groups, split): (B, H, Sq, Skv) on 256 CUs
NARROW = {(64, 4, False): (2, 1, 130, 700), (128, 1, False): (2, 2, 130, 130),
          (128, 2, False): (2, 40, 200, 700), (256, 1, False): (2, 22, 700, 1087),
          (256, 1, True): (2, 1, 200, 6000)}
FULL = {(128, 1, False): (2, 2, 200, 130), (128, 2, False): (2, 1, 200, 1500),
        (256, 1, False): (2, 22, 700, 700), (256, 1, True): (2, 1, 200, 3000)}
CASES = [(d, want, size) for dims, table in (((40, 56, 64), NARROW),
                                             ((72, 88, 104, 120, 128), FULL))
         for d in dims for want, size in table.items()]


@pytest.fixture(scope="module")
def sp():
  if not torch.cuda.is_available():
    pytest.skip("no GPU")
  if torch.cuda.get_device_properties(0).multi_processor_count != 256:
    pytest.skip("the sizes choose their shapes on 256 CUs")
  from diffusers_tpu_amd.kernels import splash
  return splash


@pytest.mark.parametrize("d,want,size", CASES,
                         ids=[f"{d}-{w}" for d, w, _ in CASES])
def test_shape_matches_oracle(sp, d, want, size):
  from diffusers_tpu_amd.kernels.block_sizes import launch_shape
  banner(f"shape {want} dim {d} {size}")
  b, h, sq, skv = size
  s = launch_shape(b, h, sq, skv, d)
  assert (s.block_rows, s.key_groups, s.split_parts > 1) == want
  assert sp._split_bytes(b, h, sq, skv, 0, d, 0) == s.workspace_bytes
  q, k, v = (seeded((b, h, n, d), 700 + i) for i, n in enumerate((sq, skv, skv)))
  heads = sorted({0, h - 1})
  rows = np.unique(np.r_[0:40, 120:136, max(0, sq - 70):sq])
  rows = rows[rows < sq]
  for lens in (None, (skv - 29, 50)):
    n = None if lens is None else torch.tensor(lens, device="cuda",
                                               dtype=torch.int32)
    got = sp.attention(q, k, v, kv_len=n)
    o, m, l = sp.residual_attention(q, k, v, kv_len=n)
    for i in range(b):
      w = A.attention_f64(to64(q[i:i + 1, heads][:, :, rows]),
                          to64(k[i:i + 1, heads]), to64(v[i:i + 1, heads]),
                          kv_len=skv if lens is None else lens[i])
      pick = lambda t: to64(t[i:i + 1, heads][:, :, rows])
      assert_attn_close(pick(got), w, f"{lens} sample {i}")
      assert_attn_close(pick(o) / pick(l), w, f"{lens} residual {i}")
    if d == 128:
      packed = sp.pack_v(v, n)
      assert torch.equal(sp._launch(q, k, v, None, n, packed_v=packed), got)


@pytest.mark.parametrize("d", [64, 128])
def test_smaller_workgroups_take_no_workspace(sp, d):
  """Calls that run in smaller workgroups hold no split buffer; reserve still
  sizes the one that an E4M3 call of the shape uses."""
  banner(f"workspace of small shapes, dim {d}")
  q = seeded((1, 8, 500, d), 710)
  ws = sp.AttentionWorkspace()
  want = sp.attention(q, q, q)
  assert torch.equal(sp.attention(q, q, q, workspace=ws), want)
  assert ws._split is None or ws._split.numel() <= 4
  ws.reserve(q.shape, q.shape)
  held = ws._split
  assert held.numel() > 4
  if d == 128:
    sp.attention(q, q, q, qk_fp8=True, workspace=ws)
    assert ws._split is held


@pytest.mark.parametrize("d,size", [(64, (2, 1, 130, 700)), (64, (2, 8, 1000, 1024)),
                                    (128, (2, 1, 200, 1500)), (128, (1, 3, 300, 4096))])
def test_no_workspace_gives_the_bits_of_the_plain_entry(sp, d, size):
  """dt_flash_fwd_ex without a workspace sweeps a block's tiles in one order,
  as dt_flash_fwd does, also where attention() uses key groups or a split."""
  from diffusers_tpu_amd import _lib
  banner(f"no workspace, dim {d} {size}")
  b, h, sq, skv = size
  q, k, v = (seeded((b, h, n, d), 720 + i) for i, n in enumerate((sq, skv, skv)))
  lib = _lib.load()
  s3 = lambda t: _lib.i64_array(*t.stride()[:3])
  st = torch.cuda.current_stream().cuda_stream
  x, y = torch.empty_like(q), torch.empty_like(q)
  scale = d ** -0.5
  _lib.check("dt_flash_fwd", lib.dt_flash_fwd(
      q.data_ptr(), k.data_ptr(), v.data_ptr(), x.data_ptr(), b, h, h, sq, skv,
      d, s3(q), s3(k), s3(v), s3(x), scale, 0, None, None, None, None, st))
  _lib.check("dt_flash_fwd_ex", lib.dt_flash_fwd_ex(
      q.data_ptr(), k.data_ptr(), 0, v.data_ptr(), s3(v), None, 0, y.data_ptr(),
      b, h, h, sq, skv, d, s3(q), s3(k), s3(y), scale, 0, None, None, None,
      None, None, None, None, None, 0, st))
  assert torch.equal(x, y)
  # the Python layer's routes take one shape: plain, and with an output given
  want = sp.attention(q, k, v)
  assert not torch.equal(want, x)
  assert torch.equal(sp.attention(q, k, v, out=torch.empty_like(q)), want)


def test_a_workspace_keeps_one_view_of_each_buffer(sp):
  banner("workspace views")
  ws = sp.AttentionWorkspace()
  for n in (100, 50, 400, 10, 400):
    view = ws.split(4 * n)
    assert view.numel() == n and view.data_ptr() == ws._split.data_ptr()
    assert ws.packed_v(n).numel() == n
  assert len(ws._views) == 2 and ws._split.numel() == 400
