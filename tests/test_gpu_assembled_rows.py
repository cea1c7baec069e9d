"""Row-wise assembly of the P1 operator (csrc/assembled_rows.hip) against the
hash-table assembly of the same stencil: identical sparsity and values within
the rounding of a reordered sum of positive terms. A site sums at most
cells x 64 products of nonnegative factors, each of at most 6 roundings, so
two orders differ by less than 2 (cells * 64 + 6) eps relatively, entry by
entry; the meshes have at most 40 cells around a node."""
import numpy as np
import pytest
import torch

from oracle import fe as ofe
from afsi_gpu_amd import _abi, workloads
from afsi_gpu_amd.mac.assembled import AssembledTransfer
from afsi_gpu_amd.mac.fe import FEGeometry
from afsi_gpu_amd.mac.grid import MACGrid
from afsi_gpu_amd.mac.transfer import from_points

pytestmark = pytest.mark.gpu
TOL = 2 * (40 * 64 + 6) * 2.3e-16


def geometry_of(which, gpu):
    t = lambda a, dtype=torch.float64: torch.tensor(np.ascontiguousarray(a), device=gpu, dtype=dtype)
    if which == 'lv':
        X, cells, values, weights = workloads.lv_p1(nt=1, ntheta=12, nphi=18)
        return FEGeometry(t(cells, torch.int64), t(values), t(weights), len(X)), t(X)
    if which == 'solid':
        X, cells = ofe.box_tets(2, (.3, .35, .4), (.7, .65, .75))
        g = ofe.p1_solid(X, cells)
    else:
        X, cells = ofe.icosphere(1, .25, (.5, .5, .5))
        g = ofe.p1_surface(X, cells)
    return FEGeometry(t(g.cells, torch.int64), t(g.values), t(g.weights), len(X)), t(X)


# finest boxes: rows below 512 sites; LV cells spanning many faces: rows of
# thousands of sites and 64 bases per cell; the last grid's rows exceed LDS
@pytest.mark.parametrize('which,shape,rows', [('solid', (16, 18, 20), True), ('sphere', (24, 16, 21), True),
                                              ('lv', (48, 48, 48), True), ('solid', (33, 70, 47), True),
                                              ('lv', (80, 72, 88), True), ('solid', (128, 120, 96), False)])
def test_rows_match_the_hash_table(gpu, which, shape, rows):
    geometry, x = geometry_of(which, gpu)
    grid = MACGrid(shape, (1., 1., 1.))
    tr = AssembledTransfer(grid, geometry)
    stencil = from_points(tr.interaction_points(x), grid)
    got = tr._rows(stencil.base, stencil.phi)
    assert (got is not None) == rows
    if not rows:
        st = tr.prepare(x)
        assert all(c['hash_attempts'] > 0 for c in st.assembly['components'])
        return
    want = tr._hashed(stencil.base, stencil.phi)
    again = tr._rows(stencil.base, stencil.phi)
    for c in range(3):
        for side in range(2):
            a, b, r = got[side][c], want[side][c], again[side][c]
            assert torch.equal(a.row_ptr, b.row_ptr) and torch.equal(a.cols, b.cols)
            assert float(((a.vals - b.vals).abs() / b.vals.abs()).max()) < TOL
            assert torch.equal(a.vals, r.vals) and a.rows == b.rows
        assert got[2][c]['raw_cell_entries'] == want[2][c]['raw_cell_entries']
        assert got[2][c]['nnz'] == want[2][c]['nnz']


def test_rows_refuse_what_the_table_refused(gpu):
    geometry, x = geometry_of('lv', gpu)
    grid = MACGrid((48, 48, 48), (1., 1., 1.))
    tr = AssembledTransfer(grid, geometry)
    nnz = tr.prepare(x).assembly['total_nnz']
    assert AssembledTransfer(grid, geometry, max_entries=nnz).prepare(x).assembly['total_nnz'] == nnz
    with pytest.raises(RuntimeError, match='budget exceeded'):
        AssembledTransfer(grid, geometry, max_entries=nnz - 1).prepare(x)
    stencil = from_points(tr.interaction_points(x), grid)
    stencil.phi[1, 77, 2, 1] = float('inf')
    with pytest.raises(FloatingPointError, match='nonfinite'):
        tr._rows(stencil.base, stencil.phi)
    stencil.base[2, 5, 0] = -1
    with pytest.raises(ValueError, match='stencil box'):
        tr._rows(stencil.base, stencil.phi)


def test_operator_without_entries(gpu):
    """Weights of zero leave no entries: preparing succeeds, as through the table."""
    geometry, x = geometry_of('solid', gpu)
    tr = AssembledTransfer(MACGrid((16, 18, 20), (1., 1., 1.)), geometry)
    geometry.weights.zero_()
    st = tr.prepare(x)
    assert st.assembly['total_nnz'] == 0
    assert all(int(m.row_ptr[-1]) == 0 and m.row_ptr.numel() == m.rows + 1 for m in st.gather + st.spread)


def test_scratch_of_few_point_cells(gpu):
    """The chunk lists follow the points per cell: for 4-point tetrahedra they
    take 96 bytes per cell, a twelfth of the stencil tables' 1152."""
    X, cells = ofe.box_tets(20, (.3, .35, .4), (.7, .65, .75))
    g = ofe.p1_solid(X, cells)
    t = lambda a, dtype=torch.float64: torch.tensor(np.ascontiguousarray(a), device=gpu, dtype=dtype)
    geometry, x = FEGeometry(t(g.cells, torch.int64), t(g.values), t(g.weights), len(X)), t(X)
    grid = MACGrid((32, 32, 32), (1., 1., 1.))
    tr = AssembledTransfer(grid, geometry)
    stencil = from_points(tr.interaction_points(x), grid)
    sizes = []
    call = _abi.call

    def counting(name, *args):
        if name == 'afsi_p1_row_boxes_f64':
            sizes.append(torch.cuda.memory_allocated() - base)
        call(name, *args)

    E, N = len(g.cells), len(X)
    _abi.call = counting
    try:
        torch.cuda.synchronize()
        base = torch.cuda.memory_allocated()
        assert tr._rows(stencil.base, stencil.phi) is not None
    finally:
        _abi.call = call
    # boxes of cells (72 B) and rows (72 B), two int64 per row and component, the chunk lists; 512 B per allocation
    assert sizes[0] <= E * (72 + 96) + N * (72 + 48) + 6 * 512
