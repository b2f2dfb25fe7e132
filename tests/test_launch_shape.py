"""What a call launches (dt_flash_fwd_shape): the choice by shape on a device
of 256 CUs, the workspace it uses, and the forms that keep 256-row blocks.  No
GPU is needed."""
import pytest

from diffusers_tpu_amd import _lib
from diffusers_tpu_amd.kernels import block_sizes as bs


def shape(*args, **kw):
  return bs.launch_shape(*args, compute_units=256, **kw)


def test_shapes_of_the_models_layers():
  s = shape(1, 8, 1024, head_dim=64)       # plumbing layer: 4 key groups
  assert (s.block_rows, s.key_groups, s.split_parts) == (64, 4, 1)
  assert (s.query_blocks, s.key_tiles, s.workspace_bytes) == (128, 16, 16)
  s = shape(2, 24, 512)                    # text refiner: 128-row blocks
  assert (s.block_rows, s.key_groups, s.workspace_bytes) == (128, 1, 0)
  s = shape(1, 40, 48360, 512)             # cross-attention
  assert (s.block_rows, s.key_groups, s.workspace_bytes) == (128, 1, 0)
  s = shape(2, 24, 4608, kv_len=4396)      # 864 blocks, the last 96 in 2 parts
  assert (s.block_rows, s.split_parts, s.tail_blocks) == (256, 2, 96)
  assert s.workspace_bytes == 96 * 2 * 256 * 130 * 4
  s = shape(1, 5, 350784)                  # 6855 blocks, the last 199 in 9
  assert (s.query_blocks, s.split_parts, s.tail_blocks) == (6855, 9, 199)
  s = shape(1, 16, 9000, head_dim=256)     # 128-row blocks, 32-key tiles
  assert (s.block_rows, s.key_tiles) == (128, 282) and s.split_parts > 1


@pytest.mark.parametrize("d", [8, 40, 64, 72, 104, 128, 136, 256])
def test_workspace_limits(d):
  """What a call takes is enough for it; with less it splits into fewer parts
  or not at all, and without any it keeps one order of tiles."""
  for b, h, sq, skv in [(1, 1, 1, 1), (1, 8, 1024, 1024), (2, 24, 512, 512),
                        (1, 3, 700, 1500), (1, 40, 9000, 512),
                        (2, 22, 700, 700), (1, 2, 300, 4096)]:
    s = shape(b, h, sq, skv, d)
    assert s.query_blocks == b * h * -(-sq // s.block_rows)
    if s.block_rows < 256 and d <= 128:
      assert (s.split_parts, s.workspace_bytes) == (1, 16 * (s.key_groups > 1))
    else:
      assert (s.workspace_bytes > 0) == (s.split_parts > 1)
    assert s == shape(b, h, sq, skv, d, workspace_bytes=s.workspace_bytes)
    none = shape(b, h, sq, skv, d, workspace_bytes=0)
    assert (none.key_groups, none.split_parts, none.workspace_bytes) == (1, 1, 0)
    if s.split_parts > 1:
      t = shape(b, h, sq, skv, d, workspace_bytes=s.workspace_bytes - 1)
      assert t.workspace_bytes < s.workspace_bytes


def test_tile_calls_keep_256_row_blocks():
  for kw in (dict(qk_fp8=True), dict(tile_table=True)):
    for d in (64, 72, 128):  # (zero-padded to 128)
      s = shape(1, 8, 1024, head_dim=d, **kw)
      assert (s.block_rows, s.key_groups, s.split_parts) == (256, 1, 4)
      assert s.workspace_bytes == 32 * 4 * 256 * 130 * 4
    with pytest.raises(NotImplementedError):
      shape(1, 8, 1024, head_dim=136, **kw)
  with pytest.raises(NotImplementedError):
    shape(1, 8, 1024, head_dim=264)
  with pytest.raises(ValueError):
    shape(1, 8, 1024, kv_len=1025)


def test_bad_arguments():
  import ctypes
  lib = _lib.load()
  out, need = (ctypes.c_int32 * 6)(), ctypes.c_size_t(0)
  for bad in ((1, 8, 64, 64, 0, 128, 2, 0, 256), (1, 8, 64, 64, 0, 128, 0, 0, -1),
              (1, 8, 64, 64, 0, 12, 0, 0, 256), (1, 8, 64, 64, 0, 64, 1, 0, 256),
              (0, 8, 64, 64, 0, 128, 0, 0, 256)):
    assert lib.dt_flash_fwd_shape(*bad, out, ctypes.byref(need)) < 0
  assert lib.dt_flash_fwd_shape(1, 8, 64, 64, 0, 128, 0, 0, 256, None,
                                ctypes.byref(need)) == _lib.DT_ERR_ARG
