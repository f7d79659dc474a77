"""The drop-in assembly on every form of input that its row-by-row path takes or leaves to the
launches after it: bit for bit what the launches per color give. Those run under stream
capture, so the reference of each case is the same call captured into a graph."""
import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def fan(n, op, mf):
    """n tets around one edge: two rows of n elements (n >= 3: an edge of valence n)."""
    t = 2 * np.pi * np.arange(n) / n
    x = np.concatenate([[[0, 0, 0], [0, 0, 1]], np.stack([np.cos(t), np.sin(t), 0.1 * t], 1)])
    e = np.array([[1, 2, 3 + k, 3 + (k + 1) % n] for k in range(n)], np.int32).ravel()
    return mf.Mesh(x.ravel(), e, np.zeros(n + 2, np.int32), 16 * n, op,
                   coef=mf.generate_coef(op, n, 5))


def both(mf, gpu, mesh, e2e=None, row=None, col=None, e2n=None, edges=None, precision=0, coef=True):
    """(row by row, color by color) values of one call on the same buffers."""
    D = gpu.DeviceArray.from_numpy
    row = D(np.ascontiguousarray(mesh.row if row is None else row, np.int32))
    col = D(np.ascontiguousarray(mesh.col if col is None else col, np.int32))
    e2n = D(np.ascontiguousarray(mesh.elemToNode if e2n is None else e2n, np.int32))
    coord, e2e = D(mesh.coord), None if e2e is None else D(np.ascontiguousarray(e2e, np.int32))
    k = D(mesh.coef) if coef and mesh.coef is not None else None
    nnz = mesh.nnz if edges is None else edges
    values = gpu.DeviceArray(nnz * mesh.dim, np.float64)
    stream = gpu.Stream()

    def call(s):
        gpu.assembly(coord, values, row, col, e2n, e2e, mesh.nbElem, nnz, mesh.dim,
                     mesh.operatorID, mesh.colorToElem, coef=k, precision=precision, stream=s)

    got = []
    graph = gpu.Graph(stream, call)
    for run in (lambda: call(stream), lambda: graph.launch(stream)):
        values.fill(np.nan)
        gpu.synchronize()
        run()
        stream.sync()
        got.append(values.numpy())
    return got


def same(pair, what):
    assert np.array_equal(pair[0], pair[1]), what


@pytest.mark.parametrize("op,precision,edges,coef",
                         list(itertools.product((0, 1), (0, 1), (False, True), (False, True))))
def test_rows_equal_colors_cubes(mf, gpu, op, precision, edges, coef):
    # rows of 4 to 27 entries; 2: one hex; 5 and 13: more quads of rows than fit evenly
    for n, shuffle in ((2, 0), (5, 3), (13, 7), (13, 0)):
        print(f"[rows] op={op} prec={precision} e2e={edges} coef={coef} n={n}", flush=True)
        coord, e2n, code, nnz = mf.generate_cube(n, 0.25, 3, shuffle)
        m = mf.Mesh(coord, e2n, code, nnz, op, coef=mf.generate_coef(op, e2n.size // 4, 9))
        e2e = mf.create_elemToEdge(m.row, m.col, m.elemToNode) if edges else None
        same(both(mf, gpu, m, e2e, precision=precision, coef=coef), n)


@pytest.mark.parametrize("op", [0, 1])
@pytest.mark.parametrize("n", [31, 32, 33, 63, 64, 65, 97, 127])
def test_rows_of_many_elements(mf, gpu, op, n):
    # one to four chunks of 32 elements, 32 / 64 / 128 colors, rows of up to 129 entries
    m = fan(n, op, mf)
    print(f"[rows fan] op={op} n={n} colors={m.nbColors}", flush=True)
    for e2e in (None, mf.create_elemToEdge(m.row, m.col, m.elemToNode)):
        for precision in (0, 1):
            same(both(mf, gpu, m, e2e, precision=precision), n)


@pytest.mark.parametrize("op", [0, 1])
@pytest.mark.parametrize("n", [23, 24, 25, 47, 48, 49, 72, 73, 96, 120, 121, 128])
def test_rows_at_the_chunks_edges(mf, gpu, op, n):
    """A row's elements are staged 24 at a time: one full chunk to five, one element more and
    one less, and the most colors there are."""
    print(f"[rows chunks] op={op} n={n}", flush=True)
    m = fan(n, op, mf)
    for e2e in (None, mf.create_elemToEdge(m.row, m.col, m.elemToNode)):
        for precision in (0, 1):
            same(both(mf, gpu, m, e2e, precision=precision), n)


@pytest.mark.parametrize("op,n", [(0, 6), (1, 6), (0, 13), (1, 13)])
def test_rows_odd_patterns(mf, gpu, op, n):
    coord, e2n, code, nnz = mf.generate_cube(n, 0.25, 3, 11)
    m = mf.Mesh(coord, e2n, code, nnz, op, coef=mf.generate_coef(op, e2n.size // 4, 9))
    N, rng = m.nbNodes, np.random.default_rng(4)
    rows = np.split(m.col, m.row[1:-1])

    def pattern(parts):
        return np.concatenate([[0], np.cumsum([len(r) for r in parts])]).astype(np.int32), np.concatenate(parts)

    print(f"[rows odd] op={op} n={n}", flush=True)
    # columns in another order, and columns that no element touches
    row, col = pattern([rng.permutation(np.concatenate([r, [N + 5, N + 6]])) for r in rows])
    same(both(mf, gpu, m, row=row, col=col, edges=int(row[-1])), "order and extra columns")
    # a value array that goes on past the last row
    same(both(mf, gpu, m, edges=m.nnz + 77), "entries past the last row")
    # nodes that no element holds, in front, between and behind: empty rows and not; then so
    # many that the row table does not reach all ids
    for far in (2, 8):
        ids = np.sort(rng.permutation(far * N)[:N])
        parts = [np.zeros(0, np.int32)] * (far * N)
        for i, r in zip(ids, rows):
            parts[i] = (ids[r - 1] + 1).astype(np.int32)
        free = [i for i in range(far * N) if len(parts[i]) == 0]
        for i in free[::3]:
            parts[i] = np.array([i + 1], np.int32)
        row, col = pattern(parts)
        wide = mf.Mesh.__new__(mf.Mesh)
        wide.__dict__.update(m.__dict__)
        wide.coord = np.zeros((far * N, 3))
        wide.coord[ids] = m.coord.reshape(-1, 3)
        wide.coord = wide.coord.ravel()
        same(both(mf, gpu, wide, row=row, col=col, e2n=(ids[m.elemToNode - 1] + 1), edges=int(row[-1])),
             f"isolated nodes {far}")
    # a missing column, a repeated one, a missing diagonal, a replaced column, a row cut to two
    for what, f in (("missing", lambda i, r: r[r != r[1]] if i % 5 == 0 else r),
                    ("repeated", lambda i, r: np.concatenate([r, r[:2]]) if i % 7 == 0 else r),
                    ("no diagonal", lambda i, r: r[r != i + 1] if i % 4 == 0 else r),
                    ("replaced", lambda i, r: np.where(r == r[2], r[3], r) if i % 6 == 0 else r),
                    ("short", lambda i, r: r[:2] if i == 40 else r)):
        row, col = pattern([f(i, r) for i, r in enumerate(rows)])
        same(both(mf, gpu, m, row=row, col=col, edges=int(row[-1])), what)


@pytest.mark.parametrize("op,n", [(0, 5), (1, 5), (0, 13), (1, 13)])
def test_rows_odd_edges(mf, gpu, op, n):
    """elemToEdge tables that are not the pattern's own: skipped blocks and blocks sent to
    entries outside the node's row, as a coupled or condensed system sends them."""
    coord, e2n, code, nnz = mf.generate_cube(n, 0.25, 3, 11)
    m = mf.Mesh(coord, e2n, code, nnz, op, coef=mf.generate_coef(op, e2n.size // 4, 9))
    e2e = mf.create_elemToEdge(m.row, m.col, m.elemToNode)
    print(f"[rows odd edges] op={op} n={n}", flush=True)
    skipped = e2e.copy()
    skipped[::37] = -1
    same(both(mf, gpu, m, skipped), "skipped")
    # the same entries stored in reverse: no row of the pattern holds its node's blocks
    same(both(mf, gpu, m, m.nnz - 1 - e2e), "reversed")
    # entries permuted inside every row
    rng, perm = np.random.default_rng(2), np.arange(m.nnz)
    for a, b in zip(m.row[:-1], m.row[1:]):
        perm[a:b] = a + rng.permutation(b - a)
    same(both(mf, gpu, m, perm[e2e]), "permuted rows")


def times(mf, gpu, mesh, row, col, e2n):
    """ms of (row by row, color by color), without elemToEdge, the least of five calls each."""
    D = gpu.DeviceArray.from_numpy
    coord, k, row, col, e2n = D(mesh.coord), D(mesh.coef), D(row), D(col), D(e2n)
    values, stream = gpu.DeviceArray(mesh.nnz * mesh.dim, np.float64), gpu.Stream()

    def call(s):
        gpu.assembly(coord, values, row, col, e2n, None, mesh.nbElem, mesh.nnz, mesh.dim,
                     mesh.operatorID, mesh.colorToElem, coef=k, stream=s)

    graph, a, b, got = gpu.Graph(stream, call), gpu.Event(), gpu.Event(), []
    for run in (lambda: call(stream), lambda: graph.launch(stream)):
        ms = []
        for _ in range(6):
            a.record(stream)
            run()
            b.record(stream)
            stream.sync()
            ms.append(a.elapsed_ms(b))
        got.append(min(ms[1:]))
    return got


def wide_ids(mf, mesh, far, seed=4):
    """The mesh as a part that keeps the ids of a whole `far` times as large (in no order):
    (coord, row, col, elemToNode)."""
    N = mesh.nbNodes
    ids = np.random.default_rng(seed).permutation(far * N)[:N]
    order = np.argsort(ids)  # the part's nodes by their new ids
    lengths = np.zeros(far * N, np.int64)
    lengths[ids] = np.diff(mesh.row)
    row = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    col = np.concatenate([ids[mesh.col[mesh.row[i]:mesh.row[i + 1]] - 1] + 1 for i in order])
    coord = np.zeros((far * N, 3))
    coord[ids] = mesh.coord.reshape(-1, 3)
    return coord.ravel(), row, col.astype(np.int32), (ids[mesh.elemToNode - 1] + 1).astype(np.int32)


@pytest.mark.parametrize("op,far", [(0, 5), (1, 5), (1, 40)])
def test_rows_of_a_part_that_keeps_global_ids(mf, gpu, op, far):
    """Ids far past a quarter of the entries are valid input: they get the same values as from
    one launch per color, and not more slowly."""
    print(f"[rows wide] op={op} far={far}", flush=True)
    coord, e2n, code, nnz = mf.generate_cube(30, 0.25, 3, 11)
    m = mf.Mesh(coord, e2n, code, nnz, op, coef=mf.generate_coef(op, e2n.size // 4, 9))
    wide = mf.Mesh.__new__(mf.Mesh)
    wide.__dict__.update(m.__dict__)
    wide.coord, row, col, e2n = wide_ids(mf, m, far)
    assert e2n.max() > m.nnz // 4 + 1
    same(both(mf, gpu, wide, row=row, col=col, e2n=e2n), f"ids {far}")
    rows, colors = times(mf, gpu, wide, row=row, col=col, e2n=e2n)
    print(f"  rows {rows:.3f} ms, colors {colors:.3f} ms", flush=True)
    assert rows < 2 * colors


def serial(mf, gpu, orc, m, e2n, e2e=None, precision=0):
    """(mf_assembly, the oracle's serial loop) with these elements and positions."""
    D = gpu.DeviceArray.from_numpy
    values = D(np.full(m.nnz * m.dim, np.nan))
    gpu.assembly(D(m.coord), values, D(m.row), D(m.col), D(e2n), None if e2e is None else D(e2e),
                 m.nbElem, m.nnz, m.dim, m.operatorID, m.colorToElem, coef=D(m.coef),
                 precision=precision)
    return values.numpy(), orc.assembly(m.coord, m.row, m.col, e2n, m.operatorID, coef=m.coef,
                                        e2e=e2e, mixed=precision != 0)


@pytest.mark.parametrize("op,precision,n", [(0, 0, 4), (1, 0, 9), (0, 1, 9), (1, 1, 4)])
def test_left_calls_equal_the_serial_loop(mf, orc, gpu, op, precision, n):
    """What the rows leave is summed in the order of the serial loop: elements that repeat a
    vertex, and an elemToEdge of reversed entries."""
    print(f"[left] op={op} precision={precision} n={n}", flush=True)
    coord, e2n, code, nnz = mf.generate_cube(n, 0.25, 3, 11)
    m = mf.Mesh(coord, e2n, code, nnz, op, coef=mf.generate_coef(op, e2n.size // 4, 9))
    e2e = mf.create_elemToEdge(m.row, m.col, m.elemToNode)
    repeats = m.elemToNode.copy()
    repeats[3::4 * 7] = repeats[2::4 * 7]
    for what, nodes, at in (("repeated vertices", repeats, None),
                            ("repeated vertices, elemToEdge", repeats,
                             mf.create_elemToEdge(m.row, m.col, repeats)),
                            ("reversed entries", m.elemToNode, m.nnz - 1 - e2e)):
        got, want = serial(mf, gpu, orc, m, nodes, at, precision)
        assert np.array_equal(got, want, equal_nan=True), what


def test_left_call_uses_the_whole_gpu(mf, gpu):
    """One element that repeats a vertex does not make the call tens of times slower."""
    coord, e2n, code, nnz = mf.generate_cube(30, 0.25, 3, 11)
    m = mf.Mesh(coord, e2n, code, nnz, 1, coef=mf.generate_coef(1, e2n.size // 4, 9))
    e2n = m.elemToNode.copy()
    e2n[3] = e2n[2]
    left, colors = times(mf, gpu, m, row=m.row, col=m.col, e2n=e2n)
    print(f"[left] {left:.3f} ms, colors {colors:.3f} ms", flush=True)
    assert left < 4 * colors


def test_large_lap_with_edges(mf, gpu):
    """The first sizes that leave the rows for the launches per color (2.5 million elements)."""
    print("[rows large]", flush=True)
    coord, e2n, code, nnz = mf.generate_cube(76, 0.25, 3, 11)
    m = mf.Mesh(coord, e2n, code, nnz, 0, coef=mf.generate_coef(0, e2n.size // 4, 9))
    D = gpu.DeviceArray.from_numpy
    dm = [D(x) for x in (m.coord, m.row, m.col, m.elemToNode, m.coef)]
    e2e, values = D(mf.create_elemToEdge(m.row, m.col, m.elemToNode)), D(np.full(m.nnz, np.nan))
    got = []
    for edges in (None, e2e):
        values.fill(np.nan)
        gpu.assembly(dm[0], values, dm[1], dm[2], dm[3], edges, m.nbElem, m.nnz, 1, 0, m.colorToElem,
                     coef=dm[4])
        got.append(values.numpy())
    same(got, "76^3")


@pytest.mark.parametrize("edges", [False, True])
def test_workspace_is_what_the_header_says(mf, gpu, edges):
    """1.5 bytes an entry and color (of 32), with elemToEdge 4 an entry more, and what the pool
    keeps is given back on request."""
    print(f"[workspace] edges={edges}", flush=True)
    coord, e2n, code, nnz = mf.generate_cube(40, 0.25, 3, 11)
    m = mf.Mesh(coord, e2n, code, nnz, 0)
    assert m.nbColors <= 32
    dm = gpu.DeviceMesh(m, with_elem_to_edge=edges)
    gpu.workspace_release()
    assert gpu.workspace_bytes() == 0
    dm.iterate_colored()
    used = (48 + (4 if edges else 0)) * m.nnz
    assert 0.8 * used < gpu.workspace_bytes() < used + (4 << 20)  # the pool's own rounding
    gpu.workspace_release()
    assert gpu.workspace_bytes() == 0
