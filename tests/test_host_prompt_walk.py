"""Where the prompt matmul's loads end, computed by the library with the functions its kernel walks by: the last row tile of a matrix may
end with its allocation, and the scalar offset that carries the walk is not bounds-checked by the hardware."""
import ctypes as C

import pytest

from turbospark_amd import ffi


def _reach(dtype, k, splits, part, rows):
    out = (C.c_int64 * 4)()
    ffi.check(ffi.lib().tsv_prompt_walk_reach(dtype, C.c_int64(k), splits, part, rows, out))
    return list(out)


# one chunk of K, a few, an odd count, many; every form of tile (64, 128, 256 rows), every part of K
@pytest.mark.parametrize("dtype,unit", [(ffi.Q4_K, 256), (ffi.Q5_K, 256), (ffi.Q6_K, 256), (ffi.Q8_0, 128), (ffi.BF16, 64), (ffi.MXFP4, 32)])
@pytest.mark.parametrize("rows", [1, 64, 65, 128, 129, 256])
def test_no_load_reaches_past_a_tile_or_a_row_block(dtype, unit, rows):
    for units in (1, 2, 3, 5, 16, 45, 90):
        chunks = -(-units * unit // (256 if dtype == ffi.MXFP4 else unit))
        for splits in (1, 2, 3, 8):
            per = -(-chunks // splits)
            if -(-chunks // per) != splits:
                continue
            for part in range(splits):
                w, w_end, a, a_end = _reach(dtype, units * unit, splits, part, rows)
                assert 0 < w <= w_end and 0 < a <= a_end, (units, splits, part)
            assert w == w_end            # (the last part's walk does reach the end)
