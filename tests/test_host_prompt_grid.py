"""The order of a prompt matmul's workgroups, by the function that the kernel and its launcher share: every (part of K, column block, row tile) once."""
import ctypes as C

import pytest

from turbospark_amd import ffi


# one column block (a router), fewer than eight, multiples of eight and not, one part of K and several, with and without a short last row tile
@pytest.mark.parametrize("short", [0, 1])
@pytest.mark.parametrize("nt,splits,mt", [(1, 1, 1), (1, 8, 16), (2, 3, 4), (7, 1, 3), (8, 5, 2), (23, 2, 6), (24, 1, 5), (40, 3, 12), (225, 1, 8)])
def test_every_tile_has_one_workgroup(nt, splits, mt, short):
    lib, out = ffi.lib(), (C.c_int32 * 5)()
    ffi.check(lib.tsv_prompt_grid(nt, splits, mt, short, 0, out))
    blocks, seen, last_full, first_short, on_die = out[0], set(), -1, None, [0] * 8
    for b in range(blocks):
        ffi.check(lib.tsv_prompt_grid(nt, splits, mt, short, b, out))
        live, split, nb, mb = out[1:]
        if not live:
            continue
        assert 0 <= split < splits and 0 <= nb < nt and 0 <= mb < mt
        assert (split, nb, mb) not in seen
        seen.add((split, nb, mb))
        on_die[b % 8] += 1
        if short and mt > 1 and mb == mt - 1:
            first_short = b if first_short is None else first_short
        else:
            last_full = b
    assert len(seen) == nt * splits * mt
    assert first_short is None or first_short > last_full
    assert max(on_die) - min(on_die) <= mt       # the units go round the dies: none has more than one unit above another
