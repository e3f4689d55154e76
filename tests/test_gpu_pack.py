"""Pack / unpack / remove on the GPU: the reference's known answers
(SparseGridGpu_tests.cu:1379-1934), packed bytes identical to the oracle's, and unpacked
grids in the same state as the oracle's."""
import numpy as np
import pytest

from tests import scenarios as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import torch
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    from openfpm_data_amd import SparseGridGpu
    return SparseGridGpu


def test_pack_known_answers_and_bytes(G, oracle):
    g, s = S.sphere_grid(G)
    o, _ = S.sphere_grid(oracle.SparseGridCpu)
    boxes = [((0, 0, 0), (321, 999, 999)), ((322, 0, 0), (999, 999, 999))]
    assert g.pack_size(boxes, [0]) == o.pack_size(boxes, [0])
    buf = g.pack(boxes, [0])
    assert S.pack_section_counts(buf, 4) == [(4685, 185807), (4475, 176787)]
    np.testing.assert_array_equal(buf, o.pack(boxes, [0]))
    # into a device buffer, and with 4-byte chunk ids
    import torch
    d = torch.zeros(len(buf) + 64, dtype=torch.uint8, device="cuda")
    n = g.pack(boxes, [0], out=d)
    np.testing.assert_array_equal(d[:n].cpu().numpy(), buf)
    np.testing.assert_array_equal(g.pack(boxes, [0], index_bytes=4), o.pack(boxes, [0], index_bytes=4))
    g.close()
    o.close()


def test_remove_sections(G, oracle):
    secs = [((310, 0, 0), (330, 999, 999)), ((0, 310, 0), (999, 330, 999)), ((0, 0, 310), (999, 999, 330))]
    grids = []
    for cls in (G, oracle.SparseGridCpu):
        g, s = S.sphere_grid(cls)
        for lo, hi in secs:
            g.remove_box(lo, hi)
        g.remove_add_unpack_finalize([])
        grids.append(g)
    S.assert_same_state(grids[0], grids[1], exist_only=False)
    p = S.existing_points(grids[0])
    for lo, hi in secs:
        assert not S.in_box(p, lo, hi).any()


def test_pack_unpack_known_counts(G, oracle):
    state = []
    for cls in (G, oracle.SparseGridCpu):
        src, s = S.sphere_grid(cls, vector=True)
        dst = cls(3, s["size"], [np.float32] * 4, block_edge=4)
        buf = S.pack_unpack_round(dst, src)
        assert S.pack_section_counts(buf, 16) == [(1107, 41003), (1420, 54276), (610, 20828), (739, 27283)]
        p = S.existing_points(dst)
        assert [int(S.in_box(p, lo, hi).sum()) for lo, hi in S.PACK_DST_BOXES] == [41003, 54276, 20828, 27283]
        sp = S.existing_points(src)
        src.remove_points(src.lin_id(sp[(sp.sum(axis=1) % 2) == 0]))
        buf2 = S.pack_unpack_round(dst, src)
        p = S.existing_points(dst)
        assert [int(S.in_box(p, lo, hi).sum()) for lo, hi in S.PACK_DST_BOXES] == [20520, 27152, 10423, 13649]
        for k, (lo, hi) in enumerate(S.PACK_DST_BOXES):
            assert S.shell_in_dst_box(p[S.in_box(p, lo, hi)], s["centre"], k).all()
        state.append((buf, buf2, dst, src))
    np.testing.assert_array_equal(state[0][0], state[1][0])
    np.testing.assert_array_equal(state[0][1], state[1][1])
    S.assert_same_state(state[0][2], state[1][2])
    S.assert_same_state(state[0][3], state[1][3], exist_only=False)


@pytest.mark.parametrize("seed", range(6))
def test_pack_unpack_random(G, oracle, seed):
    """Random grids (2D/3D, edges 2/4/8, mixed types), random boxes and property subsets:
    packed bytes equal, unpacked with a random shift into a grid that already holds points
    (one destination box removed first): same state as the oracle."""
    rng = np.random.default_rng(900 + seed)
    dim = 3 if seed % 2 else 2
    edge = [2, 4, 8][seed % 3]
    size = [int(rng.integers(3 * edge, 8 * edge)) for _ in range(dim)]
    dtypes = [[np.float64, np.int32], [np.float32, np.uint8, np.int64], [np.uint16, np.float64]][seed % 3]
    steps = S.random_flush_program(seed, dim, edge, size, dtypes, nflush=2, nrec=300)
    props = sorted(rng.choice(len(dtypes), size=int(rng.integers(1, len(dtypes) + 1)), replace=False).tolist())
    boxes = []
    for _ in range(3):
        lo = [int(rng.integers(0, s // 2)) for s in size]
        hi = [int(rng.integers(l, s)) for l, s in zip(lo, size)]
        boxes.append((lo, hi))
    res = []
    for cls in (G, oracle.SparseGridCpu):
        src = S.run_flush_program(cls, dim, edge, size, dtypes, steps)
        dst = S.run_flush_program(cls, dim, edge, size, dtypes, steps[:1])
        buf = src.pack(boxes, props, index_bytes=[4, 8][seed % 2])
        dst.remove_box(boxes[0][0], boxes[0][1])
        at = 0
        for lo, hi in boxes:
            ext = [h - l for l, h in zip(lo, hi)]
            dlo = np.minimum(np.array(lo) + 1, np.array(size) - 1 - np.array(ext)).tolist()
            at += dst.unpack(buf, dlo, props, index_bytes=[4, 8][seed % 2], offset=at)
        dst.remove_add_unpack_finalize(props)
        res.append((buf, dst))
    np.testing.assert_array_equal(res[0][0], res[1][0])
    S.assert_same_state(res[0][1], res[1][1])


@pytest.mark.parametrize("seed,props", [(0, (0,)), (1, (0, 1)), (2, (1,))])
def test_copy_to_ring(G, oracle, seed, props):
    """copy_to between three grids (one copying into itself, one removing a box), phases
    0, 1, 2 on every grid: the same grids as the oracle's."""
    res = [S.copy_ring(cls, seed, props)[0] for cls in (G, oracle.SparseGridCpu)]
    for a, b in zip(*res):
        S.assert_same_state(a, b, exist_only=False)
        a.close()
        b.close()


@pytest.mark.parametrize("dim,edge,lin", [(3, 4, "smb"), (3, 8, "zmb"), (2, 4, "smb")])
def test_links_match_oracle(G, oracle, dim, edge, lin):
    """construct_link_dw / construct_link_up: padding points, offsets and links equal the
    oracle's, both directions."""
    res = []
    for cls in (G, oracle.SparseGridCpu):
        c, f = S.link_levels(cls, 11, dim, edge, lin)
        box = ((0, 1, 0)[:dim], (19, 22, 15)[:dim])
        c.construct_link(f, 0, box, (1, 0, 1)[:dim])
        f.tag_boundaries()
        f.construct_link(c, 1, tuple(tuple(2 * v for v in b) for b in box), (0, 1, 1)[:dim])
        res.append((c.links(0), f.links(1)))
        c.close()
        f.close()
    for a, b in zip(res[0][0] + res[0][1], res[1][0] + res[1][1]):
        np.testing.assert_array_equal(a, b)
    assert len(res[0][0][3]) > 0 and len(res[0][1][3]) > 0


def test_unpack_outside_grid_fails(G):
    from openfpm_data_amd._capi import SgError
    g = G(3, (32, 32, 32), [np.float32], block_edge=8)
    g.insert_coords([[30, 30, 30]], [np.array([1.0], np.float32)])
    g.flush(["smax"])
    buf = g.pack([((28, 28, 28), (31, 31, 31))], [0])
    with pytest.raises(SgError):
        g.unpack(buf, (30, 30, 30), [0])  # the point would land at 32
    assert g.pending_inserts() == 0
    g.close()


@pytest.mark.parametrize("nbox,dim,edge,lin,index_bytes", [(1, 3, 8, "smb", 8), (8, 3, 8, "smb", 4), (9, 3, 5, "smb", 8),
                                                           (32, 2, 16, "smb", 8), (33, 3, 8, "zmb", 4), (70, 2, 6, "smb", 8)])
def test_many_boxes(G, oracle, nbox, dim, edge, lin, index_bytes):
    """Counts of boxes about what one launch and the pinned words take, chunk edges that are
    no power of two, Morton ids, value arrays at every alignment, a device buffer at an odd
    address: the oracle's bytes, and after unpacking and removing them its grid."""
    import torch
    rng = np.random.default_rng(nbox)
    size = [int(rng.integers(5 * edge, 9 * edge)) for _ in range(dim)]
    dtypes = [np.uint8, np.float64, np.uint16, np.float32]
    pts = np.stack([rng.integers(0, s, 4000) for s in size], 1).astype(np.int32)
    vals = [rng.integers(0, 200, 4000).astype(t) for t in dtypes]
    boxes = []
    for k in range(nbox):
        lo = [int(rng.integers(0, s - 1)) for s in size]
        boxes.append((lo, [int(rng.integers(l, min(s, l + 3 * edge))) for l, s in zip(lo, size)]))
    boxes[-1] = ([0] * dim, [s - 1 for s in size])
    grids = []
    for cls in (G, oracle.SparseGridCpu):
        pair = []
        for part in (slice(None), slice(0, 1500)):
            g = cls(dim, size, dtypes, block_edge=edge, linearizer=lin)
            g.insert_coords(pts[part], [v[part] for v in vals])
            g.flush(["smax"] * 4)
            pair.append(g)
        grids.append(pair)
    (a, da), (b, db) = grids
    want = b.pack(boxes, [0, 1, 2, 3], index_bytes)
    assert a.pack_size(boxes, [0, 1, 2, 3], index_bytes) == len(want)
    np.testing.assert_array_equal(a.pack(boxes, [0, 1, 2, 3], index_bytes), want)
    dev = torch.full((len(want) + 9,), 0xAB, dtype=torch.uint8, device="cuda")
    odd = dev[1:]
    assert a.pack(boxes, [0, 1, 2, 3], index_bytes, out=odd) == len(want)
    np.testing.assert_array_equal(odd.cpu().numpy()[:len(want)], want)
    assert (dev.cpu().numpy()[[0] + list(range(len(want) + 1, len(want) + 9))] == 0xAB).all()
    for g in (da, db):
        for lo, hi in boxes[:-1]:
            g.remove_box(lo, hi)
        at = 0
        for lo, _ in boxes[:-1][:12]:
            at += g.unpack(odd if g is da else want, lo, [0, 1, 2, 3], index_bytes, offset=at)
        g.remove_add_unpack_finalize([0, 1, 2, 3])
    S.assert_same_state(da, db)


def test_unpack_refuses_malformed_sections(G):
    """Chunk counts and scans that lead outside the section are refused, host and device."""
    import torch
    from openfpm_data_amd._capi import SgError
    g = G(3, (32, 32, 32), [np.float32], block_edge=8)
    g.insert_coords([[1, 2, 3], [20, 20, 20]], [np.array([1.0, 2.0], np.float32)])
    g.flush(["smax"])
    good = g.pack([((0, 0, 0), (31, 31, 31))], [0])
    head = 8 + 24
    bad = [good[:head - 1], good[:head + 17], good[:-1]]
    for at, v in ((0, 1 << 62), (0, len(good)), (0, (1 << 64) - 2)):
        x = good.copy()
        x[at:at + 8] = np.frombuffer(np.uint64(v).tobytes(), np.uint8)
        bad.append(x)
    x = good.copy()
    x[head + 16:head + 20] = 1  # the scan starts past 0
    bad.append(x)
    for x in bad:
        for buf in (x, torch.from_numpy(x.copy()).cuda()):
            with pytest.raises(SgError):
                g.unpack(buf, (0, 0, 0), [0])
    assert g.pending_inserts() == 0
    assert g.unpack(torch.from_numpy(good).cuda(), (0, 0, 0), [0]) == len(good)
    g.close()
