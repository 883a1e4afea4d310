"""The parts of K in which a matmul that leaves partial sums is cut: they fix the order of a sum, and so the bits of every row, and how many
chunks a workgroup of the 64-row passes walks one after the other."""
import pytest

from turbospark_amd import ffi

CHUNK = {12: 256, 13: 256, 14: 256, 39: 256, 8: 128, 30: 64}


# (dtype, rows, cols) -> parts: the projections of the configurations in use, and shapes beside them whose parts could be made a whole number of
# workgroups for each of 256 compute units
@pytest.mark.parametrize("dtype,rows,cols,parts", [
    (12, 4096, 4096, 4), (12, 4096, 14336, 7), (14, 4096, 14336, 7), (12, 4160, 14336, 7), (12, 8192, 8192, 2), (12, 16384, 4096, 1),
    (8, 4096, 14336, 7), (12, 6144, 4096, 4), (8, 2048, 4096, 8), (30, 2880, 4096, 8), (30, 128, 2880, 8), (8, 128, 2048, 4), (12, 64, 256, 1)])
def test_the_parts_of_k_of_a_shape(dtype, rows, cols, parts):
    assert ffi.matmul_parts(dtype, rows, cols) == parts


@pytest.mark.parametrize("dtype", sorted(CHUNK))
def test_a_part_is_about_four_waves_long(dtype):
    """A workgroup has about four waves' chunks to walk (one, two or four chunks a wave, by how much there is to spread), until eight parts are
    reached; and no part is empty."""
    for tiles in (1, 2, 7, 16, 64, 65, 128, 255, 256, 512):
        for chunks in (1, 2, 3, 8, 16, 31, 56, 57, 112, 224, 300):
            parts = ffi.matmul_parts(dtype, tiles * 64, chunks * CHUNK[dtype])
            total, per = tiles * chunks, -(-chunks // parts)
            walk = 4 if total >= 4096 else 2 if total >= 2048 else 1
            assert 1 <= parts <= 8 and (parts - 1) * per < chunks
            assert per <= 4 * walk or per == -(-chunks // 8), (tiles, chunks, parts)


def test_no_shape_at_all_is_refused():
    for bad in ((99, 64, 256), (12, 0, 256), (12, 64, 0)):
        with pytest.raises(Exception, match="bad argument"):
            ffi.matmul_parts(*bad)
