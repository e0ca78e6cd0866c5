"""Host-side checks of the element assembly plan (no GPU): coloured patches, coloured elements, atomics.

Invariants (sf2d_plan_validate): every listed element appears once in the device order; no two units
(patches or elements) of one colour share a GLL point; patch slots address their patch's point list;
patches hold at most 10 elements and 256 points; the patch mode's internal point numbering is a
permutation in which every patch owns one contiguous id range (ranges disjoint) and lists, sorted, only
points owned by other patches as its halo.  On structured meshes a 10-element strip owns its upper four
GLL rows (160 points) and reads 45 halo points (the row below and the column to its left)."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

from oracle.oracle import OracleSim
from specfem2d_amd import config, driver

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def validate(ibool, nglob, lists, mode):
    gpu, _ = driver.load_libraries()
    nspec = ibool.shape[0]
    np_ = lists.shape[1]
    ib = np.ascontiguousarray(ibool.reshape(-1), dtype=np.int32)
    ph = np.ascontiguousarray(lists.reshape(-1), dtype=np.int32)
    stats = np.zeros(6, np.int32)
    f = gpu.sf2d_plan_validate
    f.restype = C.c_int
    rc = f(C.c_int(nspec), C.c_int(nglob), ib.ctypes.data_as(C.c_void_p), C.c_int(np_),
           ph.ctypes.data_as(C.c_void_p), C.c_int(mode), stats.ctypes.data_as(C.c_void_p))
    return rc, stats


def inner_only(nspec):
    lists = np.zeros((2, nspec), np.int32)
    lists[1] = np.arange(1, nspec + 1)
    return lists


MESHES = {
    "tromp": lambda: config.tromp2005_kernel(nstep=2),
    "c1": lambda: config.plain_elastic_c1(nstep=2),
    "layers": lambda: config.small_test_mesh(nx=13, nz=10, nstep=2).replace(
        interfaces=[-1000.0, -620.0, -330.0, 0.0], nz_layers=[3, 4, 3], xmax=1390.0),
}


@pytest.mark.parametrize("name", sorted(MESHES))
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_plan_invariants_structured(name, mode):
    cfg = MESHES[name]()
    o = OracleSim(cfg, "sp")
    rc, stats = validate(o.ibool(), o.nglob, inner_only(o.nspec), mode)
    assert rc == 0
    if mode in (0, 1):
        assert stats[0] == 0 and stats[1] == 4  # 2 x 2 checkerboard of elements or of row patches
    if mode == 0:
        npatch = sum((cfg.nx + 9) // 10 for _ in range(cfg.nz))  # row segments of <= 10 elements
        assert stats[2] == npatch
        assert stats[3] <= 41 * 5
        assert stats[5] == o.nglob  # every point owned by exactly one patch
        # halo of each strip: the GLL row below it and the column to its left, where those exist
        expect = 0
        for ez in range(cfg.nz):
            for x0 in range(0, cfg.nx, 10):
                w = min(10, cfg.nx - x0)
                if ez > 0:
                    expect += 4 * w + 1 + (4 if x0 > 0 else 0)  # row below (with its corner), left column
                elif x0 > 0:
                    expect += 5  # bottom strip: the whole left column
        assert stats[4] == expect


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_plan_invariants_shuffled_and_split_lists(mode):
    # an arbitrary element order and an outer/inner split, as a partitioned mesh would pass
    cfg = config.small_test_mesh(nx=17, nz=11, nstep=2)
    o = OracleSim(cfg, "sp")
    rng = np.random.default_rng(4)
    perm = rng.permutation(o.nspec) + 1
    nout = 37
    lists = np.zeros((2, o.nspec - nout), np.int32)
    lists[0, :nout] = perm[:nout]
    lists[1, :] = perm[nout:]
    rc, stats = validate(o.ibool(), o.nglob, lists, mode)
    assert rc == 0
    if mode != 2:
        assert stats[0] >= 1 and stats[1] >= 4


def chains(ibool, nglob, lists, first=None):
    gpu, _ = driver.load_libraries()
    ib = np.ascontiguousarray(ibool.reshape(-1), dtype=np.int32)
    ph = np.ascontiguousarray(lists.reshape(-1), dtype=np.int32)
    f = gpu.sf2d_plan_chains
    f.restype = C.c_int
    nf = C.c_int(-1)
    rc = f(C.c_int(ibool.shape[0]), C.c_int(nglob), ib.ctypes.data_as(C.c_void_p), C.c_int(lists.shape[1]),
           ph.ctypes.data_as(C.c_void_p), C.byref(nf))
    if first is not None:
        first.append(nf.value)
    return rc


@pytest.mark.parametrize("nx,expect", [(80, 1), (12, 1), (13, 1), (10, 1), (8, 1), (4, 1), (3, 0), (1, 0)])
def test_chain_patches_on_structured_meshes(nx, expect):
    """Rows of elements split into strips that are chains, whether they are listed row by row or in any order; meshes
    narrower than four elements fall back to the general patch kernel.  The chain property itself is re-derived here from
    ibool: along a strip of consecutive elements of one row, element k's points (4, j) are element k+1's points (0, j)."""
    cfg = config.small_test_mesh(nx=nx, nz=4, nstep=2)
    o = OracleSim(cfg, "sp")
    ib = o.ibool()
    first = []
    assert chains(ib, o.nglob, inner_only(o.nspec), first) == expect
    # first-touch assembly: exactly one update per point is the step's first
    assert first[0] == (o.nglob if expect else 0)
    if expect:
        e = np.arange(o.nspec).reshape(cfg.nz, cfg.nx)
        left, right = e[:, 1:].reshape(-1), e[:, :-1].reshape(-1)
        b = ib.reshape(-1, 5, 5)
        np.testing.assert_array_equal(b[right][:, :, 4], b[left][:, :, 0])
    # a shuffled element list is put into rows again
    rng = np.random.default_rng(3)
    lists = inner_only(o.nspec)
    lists[1] = rng.permutation(lists[1])
    first = []
    assert chains(ib, o.nglob, lists, first) == expect
    assert first[0] == (o.nglob if expect else 0)


def row_records(ibool, nglob, lists):
    gpu, _ = driver.load_libraries()
    ib = np.ascontiguousarray(ibool.reshape(-1), dtype=np.int32)
    ph = np.ascontiguousarray(lists.reshape(-1), dtype=np.int32)
    f = gpu.sf2d_plan_row_records
    f.restype = C.c_int
    n = C.c_int(-1)
    rc = f(C.c_int(ibool.shape[0]), C.c_int(nglob), ib.ctypes.data_as(C.c_void_p), C.c_int(lists.shape[1]),
           ph.ctypes.data_as(C.c_void_p), C.byref(n))
    return rc, n.value


@pytest.mark.parametrize("nx,expect", [(80, 1), (12, 1), (13, 1), (10, 1), (8, 1), (4, 1), (3, -1)])
@pytest.mark.parametrize("shuffled", [False, True])
def test_chain_row_records(nx, expect, shuffled):
    """The column-lane kernel's point ids as one record per chain row: in the plan's numbering every GLL row of a
    chain is numbered consecutively (column x > 0 at base + x), so {base, id of column 0, first-touch mask} per row
    reproduces the id and first-touch flag of every writing lane (checked point by point on the host); meshes whose
    patches are not chains have no records."""
    cfg = config.small_test_mesh(nx=nx, nz=4, nstep=2)
    o = OracleSim(cfg, "sp")
    lists = inner_only(o.nspec)
    if shuffled:
        lists[1] = np.random.default_rng(3).permutation(lists[1])
    rc, n = row_records(o.ibool(), o.nglob, lists)
    assert rc == expect
    if expect == 1:
        assert n == 5 * -(-nx // 12) * cfg.nz


ROWS = """
import sys
import numpy as np
from tests.test_assembly_plan import chains, inner_only, validate
rows, long = {rows}, 12
# rows of twelve elements without neighbours above or below, but every two rows share one point of their top edges
g = np.arange(rows * 5 * (4 * long + 1), dtype=np.int64).reshape(rows, 5, 4 * long + 1)
for a in range(rows):
    for b in range(a):
        g[a, 4, b + 1] = g[b, 4, a + 1]
ib = np.zeros((rows, long, 5, 5), np.int64)
for k in range(long):
    ib[:, k] = g[:, :, 4 * k:4 * k + 5]
_, ib = np.unique(ib, return_inverse=True)
ib = ib.reshape(rows, long, 25) + 1
ib = np.ascontiguousarray(ib.transpose(1, 0, 2)).reshape(rows * long, 25).astype(np.int32)  # column by column
lists = inner_only(rows * long)
assert validate(ib, ib.max(), lists, 0)[0] == 0, "the general patches"
print("chains", chains(ib, int(ib.max()), lists), flush=True)
"""


@pytest.mark.parametrize("rows,expect", [(32, 1), (33, 0), (46, 0)])
def test_rows_that_need_too_many_colours_are_no_chains(rows, expect):
    """Rows can meet in more points than patches do: where 32 colours do not keep them apart, the mesh keeps the general
    patches (in a process of its own, which an error ends)."""
    out = subprocess.run([sys.executable, "-c", ROWS.format(rows=rows)], capture_output=True, text=True, cwd=ROOT)
    assert out.returncode == 0 and f"chains {expect}" in out.stdout, out.stdout + out.stderr


def test_element_arrays_beyond_4_gib():
    """Element arrays of 8 and 16 bytes a point (moduli, geometry per point) pass 4 GiB at 21.5 and 10.7 million elements,
    which a handle takes (it refuses 4 GiB of an array of 4 bytes a point, 42.9 million): their last points lie where they
    should."""
    gpu, _ = driver.load_libraries()
    f = gpu.sf2d_plan_element_byte
    f.restype = C.c_long
    for bytes_, first in ((4, 42949660), (8, 21474836), (8, 21474837), (8, 42949660), (16, 10737418), (16, 10737419),
                          (16, 42949660)):
        for k in (0, 1, 11, 16 * 12 - 1):  # a chain, and a tower of 16
            for p in (0, 24):
                assert f(bytes_, first, k, p) == bytes_ * ((first + k) * 25 + p)
