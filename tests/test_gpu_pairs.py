"""Grid builds of scenes with large triangles, whose cells are spread over the
launch in slices: waves of 64 triangles about the number of candidates from
which they are listed, every wave listed, and lists longer than one pass of the
slices' workgroups.  Cells, leaves and references equal the oracle's."""
import numpy as np
import pytest

import pyoracle as O
from gpu_util import SEED, assert_grid_equal, gpu_engine, oracle_grid
from happyray_amd import GRID_TWO_LEVEL, GRID_UNIFORM, GRID_UNIFORM_EXACT, Batch, scenes

pytestmark = pytest.mark.gpu


def walls_and_soup(seed, walls, soup, size=0.2):
    """`walls` triangles that cross most of the scene, small ones before and after."""
    sc = scenes.random_soup(seed, walls + soup, extent=10.0, size=size)
    rng = np.random.default_rng(seed)
    v = sc.verts.reshape(3, -1, 3)
    first = soup // 2
    v[:, first:first + walls] = rng.uniform(0.0, 10.0, (3, walls, 3))
    sc.verts = np.ascontiguousarray(v.reshape(3, -1)).astype(np.float32)
    return sc


# (walls, soup, density): one wall of about 1024 cells and fewer, a ground's two
# triangles among many, a wave of walls, only walls, thousands of them
SIZES = [(1, 3000, 2.0), (1, 3000, 4.0), (2, 20000, 5.0), (64, 1000, 3.0), (65, 0, 6.0), (300, 4000, 1.0),
         (4000, 0, 0.25)]


@pytest.mark.parametrize("kind", [GRID_UNIFORM, GRID_UNIFORM_EXACT, GRID_TWO_LEVEL])
@pytest.mark.parametrize("walls,soup,density", SIZES)
def test_large_triangles(kind, walls, soup, density):
    sc = walls_and_soup(walls + soup, walls, soup)
    e = gpu_engine(sc, kind, density, 2.0)
    assert_grid_equal(e, oracle_grid(sc, kind, density, 2.0))
    e.build_acc_struct()                      # again, with the buffers it has grown to
    assert_grid_equal(e, oracle_grid(sc, kind, density, 2.0))
    e.close()


def test_large_triangles_in_a_batch():
    scs = [walls_and_soup(70 + i, w, s) for i, (w, s, _) in enumerate(SIZES[:6])]
    b = Batch()
    b.set_scenes([(sc.verts, sc.idx) for sc in scs])
    b.set_densities(1.2, 2.0)
    b.build()
    for s, sc in enumerate(scs):
        og = oracle_grid(sc, GRID_TWO_LEVEL, 1.2, 2.0)
        _, cells, leaves, prims = b.grid(s)
        np.testing.assert_array_equal(cells, og.cells())
        np.testing.assert_array_equal(leaves, og.leaves())
        np.testing.assert_array_equal(prims, og.prims())
    b.close()


# triangles and density such that the cell or leaf keys have 16, 17, 19, 20 and
# 21 bits (digits of 8, 9 and 10) over few sort chunks and over more than 128
@pytest.mark.parametrize("kind,tris,density", [
    (GRID_TWO_LEVEL, 3000, 0.25), (GRID_TWO_LEVEL, 12000, 0.25), (GRID_TWO_LEVEL, 40000, 0.25),
    (GRID_TWO_LEVEL, 100000, 0.25), (GRID_TWO_LEVEL, 140000, 1.2), (GRID_UNIFORM, 20000, 20.0),
    (GRID_UNIFORM, 70000, 1.5), (GRID_UNIFORM, 1, 1.0), (GRID_UNIFORM, 681, 3.0)])
def test_sort_widths(kind, tris, density):
    sc = scenes.random_soup(tris, tris, extent=10.0, size=0.1)
    e = gpu_engine(sc, kind, density, 2.0)
    assert_grid_equal(e, oracle_grid(sc, kind, density, 2.0))
    e.close()
