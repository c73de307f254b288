"""What the selection rules can return against what is compiled, on the CPU."""
import ctypes

import pytest

from fastlstm_amd import _lib

LDS_LIMIT = 160 << 10


@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("backward", [0, 1])
def test_every_shape_of_the_xcd_local_kernels_is_compiled(dtype, backward):
    """All hidden sizes of up to 32 workgroups of 32 units, every number of batch tiles until none fits, one to four recurrences."""
    lib, shape, used = _lib.load(), (ctypes.c_int * 5)(), set()
    for H in range(16, 1040, 8):
        for copies in (1, 2, 3, 4):
            for tiles in range(1, 140):
                rc = lib.fastlstm_diag_xcd_shape(16 * tiles - 7, H, dtype, backward, copies, shape)
                assert rc in (0, 1), (H, 16 * tiles - 7, copies, tuple(shape))
                if rc:
                    assert shape[4] <= LDS_LIMIT
                    used.add(tuple(shape[:4]))
    # fp32, forward: units per workgroup 8, 16, 32, with batch tiles of 16 and 32 rows each
    if dtype == 0 and not backward:
        assert {(mt, ntw) for mt, _, ntw, _ in used} == {(mt, ntw) for mt in (2, 4, 8) for ntw in (1, 2)}


@pytest.mark.parametrize("T,B,I,H,dtype,parts", [(50, 100, 100, 512, 1, 8), (50, 100, 100, 256, 2, 4), (16, 64, 72, 2048, 1, 2), (16, 16, 64, 256, 0, 2)])
def test_the_weight_gradients_workspace_holds_the_parts_of_dx(T, B, I, H, dtype, parts):
    """Few output tiles of d.Wx and a long sum: the product is cut into that many parts at least (operands that the tile kernel takes and
    ones that it does not, I = 100), whose place is this workspace."""
    assert _lib.load().fastlstm_wgrad_workspace_bytes(T, B, I, H, dtype) >= parts * T * B * I * 4
