"""Sizes of the cone forward's bricked copy on both sides of the limits of the
tracked walk's layout (host arithmetic only)."""
import ctypes as C

import pytest

GIB = 1 << 30


def _bytes(nx, ny, nz, nt, tracked):
    from framelab_amd import _lib
    fn = getattr(_lib.lib(), "_Z18fl_cone_copy_bytesiiiib")   # size_t fl_cone_copy_bytes(int, int, int, int, bool)
    fn.restype, fn.argtypes = C.c_size_t, [C.c_int] * 4 + [C.c_bool]
    return fn(nx, ny, nz, nt, tracked)


def _padded(nx, ny, nz):
    p2 = lambda n: max(4, 1 << (n - 1).bit_length())  # noqa: E731
    return p2(nx) * p2(ny) * 4 * ((nz + 3) // 4 + 4)   # whole bricks, two guard layers below and above


@pytest.mark.parametrize("nx, ny, nz, nt, tracked", [
    (8, 8, 8, 1, True), (256, 256, 256, 1, True), (512, 512, 512, 1, True), (130, 130, 130, 1, True),
    # four times the voxels: by 4 GiB
    (514, 514, 514, 1, True), (514, 514, 994, 1, True), (514, 514, 1010, 1, False),
    # above it, where at most twice the plain copy
    (1024, 1024, 900, 1, True), (1024, 600, 900, 1, True), (1024, 500, 2000, 1, True), (1024, 514, 2000, 1, False),
    # 2^30 voxels and more
    (1024, 1024, 1008, 1, True), (1024, 1024, 1012, 1, False), (1026, 1026, 240, 1, True), (1026, 1026, 244, 1, False),
    # many thin frames
    (34, 34, 2, 13107, True), (34, 34, 2, 13108, False),
])
def test_limits(nx, ny, nz, nt, tracked):
    plain, padded = _bytes(nx, ny, nz, nt, False), _bytes(nx, ny, nz, nt, True)
    assert plain >= nx * ny * nz * nt * 4
    assert (padded > 0) == tracked
    if tracked:
        assert padded >= _padded(nx, ny, nz) * nt * 4 and padded >= plain
        assert padded <= max(4 * GIB, 2 * plain)
    else:
        assert _padded(nx, ny, nz) > GIB or _padded(nx, ny, nz) * nt * 4 > max(4 * GIB, 2 * plain)
