"""Workspace sizes of the block statistics by dtype (host only)."""
from pasa_amd import _lib


def test_workspace_bytes_dtype():
    lib = _lib.load()
    f, old = lib.pasa_block_stats_workspace_bytes_dtype, lib.pasa_block_stats_workspace_bytes
    # where the tuned head_dim 128 kernels run it is the size without a dtype
    for args in ((12, 32760, 0, 128, 128, 32), (40, 75600, 0, 128, 128, 32)):
        assert f(*args, _lib.DTYPE_BF16) == old(*args)
    assert f(12, 32760, 0, 128, 128, 32, _lib.DTYPE_F16) == old(12, 32760, 0, 128, 128, 32)
    # head_dim 64: at least four blocks to a part (eight groups of 32 blocks per slice here)
    assert f(12, 32760, 0, 64, 128, 32, _lib.DTYPE_BF16) == 12 * 8 * 8 * 64 * 64 * 4
    # and groups of 16 or more: a smaller one is done before a second launch pays
    assert f(2, 1024, 0, 64, 128, 32, _lib.DTYPE_BF16) == f(2, 959, 0, 64, 64, 32, _lib.DTYPE_BF16) == 0
    assert f(2, 1024, 0, 64, 64, 32, _lib.DTYPE_BF16) == 2 * 4 * 64 * 64 * 4
    # the any-shape kernels: a power-of-two number of parts of D x D floats per group, at most one per block
    per_group = 64 * 64 * 4
    assert f(2, 1024, 0, 64, 64, 32, _lib.DTYPE_F32) == 2 * 16 * per_group
    assert f(1, 16, 0, 64, 16, 32, _lib.DTYPE_F32) == 0          # one block: nothing to split
    assert f(600, 1024, 0, 64, 64, 32, _lib.DTYPE_F32) == 0      # enough groups already
    assert f(2, 1024, 0, 64, 64, 32, 7) == 0                     # no such dtype
    assert f(2, 1024, 0, 64, 48, 32, _lib.DTYPE_F32) == 0        # no such block size
    assert f(2, 0, 0, 64, 64, 32, _lib.DTYPE_F32) == 0
