"""GPU parity of the tiled star-stencil kernels (2D 16^2 chunks: every kind; 8^3 chunks:
red-black SOR and the residual) against the oracle, bit for bit."""
import numpy as np
import pytest

from openfpm_data_amd import _capi as C
from tests import scenarios as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import torch
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    from openfpm_data_amd import SparseGridGpu
    return SparseGridGpu


def _pair(G, oracle, dim, edge, size, dtype, seed, lin="smb", tag=True):
    """The same random grid twice (library, oracle): points dense enough for whole chunks,
    ragged enough for partial rows, padding-only points among them, background not zero."""
    rng = np.random.default_rng(seed)
    steps = S.random_flush_program(seed, dim, edge, size, [dtype] * 3, nflush=2, nrec=150, ops=["smax"] * 3)
    dense = np.stack(np.meshgrid(*[np.arange(s) for s in size], indexing="ij"), -1).reshape(-1, dim)
    dense = dense[rng.random(len(dense)) < np.where(dense[:, 0] < size[0] // 2, 1.0, 0.3)]
    vals = [rng.uniform(-1, 1, len(dense)).astype(dtype) for _ in range(3)]
    out = []
    for cls in (G, oracle.SparseGridCpu):
        g = cls(dim, size, [dtype] * 3, block_edge=edge, linearizer=lin)
        for p in range(3):
            g.set_background_value(p, p + 1)
        g.insert_coords(dense.astype(np.int32), vals)
        g.flush(["smax"] * 3)
        if lin == "smb":
            for recs, ops in steps:
                for kind, keys, masks, v in recs:
                    (g.insert if kind == "points" else g.insert_block)(*((keys, v, masks) if kind == "points" else (keys, masks, v)))
                g.flush(ops)
        g.find_neighbours(C.NN_STAR)
        if tag:
            g.tag_boundaries(C.NN_STAR)
        out.append(g)
    # padding-only slots have no specified value after a flush: start from identical arrays
    for p in range(3):
        out[1].set_prop(p, out[0].prop(p))
    return out


def _descs(rng, dim, size):
    out = []
    for apply in (C.APPLY_INTERIOR, C.APPLY_EXISTING):
        for boxed in (False, True):
            lo = [int(rng.integers(0, max(1, s // 3))) for s in size]
            box = (lo, [int(rng.integers(l, s)) for l, s in zip(lo, size)]) if boxed else None
            out += [C.make_desc(C.ST_LAP, [0], [1], apply, box, [-2.0 * dim, 1.0]),
                    C.make_desc(C.ST_LAP, [1], [1], apply, box, [-0.5, 0.125]),
                    C.make_desc(C.ST_HEAT, [1], [2], apply, box, [0.125]),
                    C.make_desc(C.ST_HEAT, [2], [2], apply, box, [0.1]),
                    C.make_desc(C.ST_GRAY_SCOTT, [0, 1], [0, 1], apply, box, [0.2, 0.1, 0.04, 0.06, 0.5]),
                    C.make_desc(C.ST_GRAY_SCOTT, [0, 1], [2, 1], apply, box, [0.2, 0.1, 0.04, 0.06, 0.5]),
                    C.make_desc(C.ST_RBSOR, [2, 0], [], apply, box, [1.3], [0]),
                    C.make_desc(C.ST_RBSOR, [2, 0], [], apply, box, [1.3], [1]),
                    C.make_desc(C.ST_RBSOR, [1, 1], [], apply, box, [0.7], [1]),
                    C.make_desc(C.ST_RESIDUAL, [2, 0], [1], apply, box),
                    C.make_desc(C.ST_RESIDUAL, [2, 0], [2], apply, box),
                    C.make_desc(C.ST_RESIDUAL, [2, 0], [0], apply, box)]
    return out


# chunk counts around the workgroups' 4 chunks (1, 3, 4, 5, 4 k + 1 and others), ragged last chunks
@pytest.mark.parametrize("lin", ["smb", "zmb"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("dim,edge,size", [(2, 16, (16, 16)), (2, 16, (130, 17)), (2, 16, (75, 91)), (2, 16, (200, 170)),
                                           (2, 16, (48, 16)), (2, 16, (30, 31)), (2, 16, (16, 77)), (2, 16, (269, 13)),
                                           (3, 8, (8, 8, 8)), (3, 8, (33, 9, 17)), (3, 8, (41, 30, 25)),
                                           (3, 8, (24, 7, 8)), (3, 8, (15, 16, 8)), (3, 8, (8, 8, 37)), (3, 8, (133, 5, 6))])
def test_star_kernels_match_the_oracle(G, oracle, dim, edge, size, dtype, lin):
    rng = np.random.default_rng(dim * 1000 + size[0])
    a, b = _pair(G, oracle, dim, edge, size, dtype, 31 + size[0], lin)
    for i, d in enumerate(_descs(rng, dim, size)):
        if lin == "smb" and dim == 3 and i % 2:
            a.set_tuning(C.TUNE_STENCIL_SKIP_EMPTY_ROWS, (i // 2) % 5)
        a.apply_stencil(d)
        b.apply_stencil(d)
        S.assert_same_state(a, b)
    # slots without a point still hold the background
    m = a.masks()
    for p in range(3):
        assert (a.prop(p)[m == 0] == p + 1).all()


@pytest.mark.parametrize("dim,edge,n", [(2, 16, 600), (3, 8, 72)])
def test_many_workgroups(G, oracle, dim, edge, n):
    """More chunks than one workgroup per XCD: the order in which they are dealt to the XCDs covers
    them all."""
    a, b = _pair(G, oracle, dim, edge, (n,) * dim, np.float32, 5, tag=False)
    for d in _descs(np.random.default_rng(1), dim, (n,) * dim)[12:]:
        a.apply_stencil(d)
        b.apply_stencil(d)
    S.assert_same_state(a, b)


@pytest.mark.parametrize("dim,edge,dtype", [(3, 8, np.float32), (3, 8, np.float64), (2, 16, np.float32)])
@pytest.mark.parametrize("nb", [1, 5, 17])
def test_chunk_runs(G, oracle, dim, edge, dtype, nb):
    """Chunks dealt to the XCDs in runs: fewer and more than the longest run takes (17^3 and
    65^2 chunks), with a last run that is not full.  Bit-exact against the oracle."""
    nb = {17: 65}.get(nb, nb) if dim == 2 else nb
    size = [nb * edge - 3] * dim
    rng = np.random.default_rng(nb)
    pts = rng.integers(0, size[0], (nb ** dim * 9, dim)).astype(np.int32)
    pts = np.concatenate([pts, pts + np.eye(dim, dtype=np.int32)[0]]).clip(0, size[0] - 1)
    vals = [rng.uniform(-1, 1, len(pts)).astype(dtype) for _ in range(3)]
    a, b = (cls(dim, size, [dtype] * 3, block_edge=edge) for cls in (G, oracle.SparseGridCpu))
    for g in (a, b):
        g.insert_coords(pts, vals)
        g.flush(["smax"] * 3)
        g.find_neighbours(C.NN_STAR)
    for d in [C.make_desc(C.ST_HEAT, [0], [2], C.APPLY_EXISTING, None, [0.1]),
              C.make_desc(C.ST_GRAY_SCOTT, [0, 1], [2, 1], C.APPLY_EXISTING, None, [0.2, 0.1, 0.04, 0.06, 0.5]),
              C.make_desc(C.ST_RBSOR, [2, 0], [], C.APPLY_EXISTING, None, [1.3], [1]),
              C.make_desc(C.ST_RESIDUAL, [2, 0], [1], C.APPLY_EXISTING, None)]:
        for g in (a, b):
            g.apply_stencil(d)
        S.assert_same_state(a, b)


@pytest.mark.parametrize("skip", [0, 1, 2, 3, 4])
def test_captured_sweeps_follow_the_masks(G, oracle, skip):
    """A sweep and a residual captured before any table of the skip modes exists, replayed after
    tags and points have changed: every replay does what the oracle does on the masks of then."""
    import torch
    a, b = _pair(G, oracle, 3, 8, (41, 30, 25), np.float64, 9, tag=False)
    s = torch.cuda.Stream()
    a.set_stream(s)
    a.set_tuning(C.TUNE_STENCIL_SKIP_EMPTY_ROWS, skip)
    descs = [C.make_desc(C.ST_RBSOR, [2, 0], [], C.APPLY_INTERIOR, None, [1.3], [0]),
             C.make_desc(C.ST_RBSOR, [2, 0], [], C.APPLY_INTERIOR, None, [1.3], [1]),
             C.make_desc(C.ST_RESIDUAL, [2, 0], [1], C.APPLY_INTERIOR)]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        for d in descs:
            a.apply_stencil(d)
    rng = np.random.default_rng(2)
    for step in range(3):
        graph.replay()
        torch.cuda.synchronize()
        for d in descs:
            b.apply_stencil(d)
        S.assert_same_state(a, b)
        if step == 0:
            for g in (a, b):
                g.tag_boundaries(C.NN_STAR)
        else:
            keys = rng.choice(a.num_chunks() * 512, 900, replace=False)
            keys = a.chunk_ids()[keys // 512] * 512 + keys % 512
            for g in (a, b):
                g.remove_points(keys)
