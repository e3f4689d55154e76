"""Batched Poisson solves on the GPU (sg_batch_* / sg_poisson_solve).

* kernel parity: one outer iteration of the mixed form equals the oracle's red-black SOR
  sweeps (FP32) and FP64 residual, bit-exact;
* convergence: mixed (FP32 sweeps + FP64 defect correction) and plain FP64 reach the
  relative residual 1e-10, re-verified with the oracle's FP64 residual on the returned u;
  the mixed solution is compared with the all-FP64 one (error bound stated below);
* continuous batching: a grid's solution is bitwise the same alone and in a mix.
"""
import numpy as np
import pytest

from openfpm_data_amd import _capi as C
from openfpm_data_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def P():
    import torch
    assert torch.cuda.is_available()
    from openfpm_data_amd import poisson
    return poisson


def _small_grids(n, seed, edge_hi=96):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(n):
        edge, occ, ids = W.random_chunk_grid(rng, 32, edge_hi)
        out.append({"size": (edge,) * 3, "chunk_ids": ids, "f": rng.uniform(-1, 1, (ids.size, 512))})
    return out


def _oracle_grid(oracle, spec, props):
    g = oracle.SparseGridCpu(3, spec["size"], props, block_edge=8)
    n = spec["chunk_ids"].size
    vals = [np.zeros((n, 512), p) for p in props]
    return g, vals


def _oracle_residual(oracle, spec, u_chunks):
    """FP64 ||f - A u|| / ||f|| with the oracle's residual stencil (u on the same chunks)."""
    g = oracle.SparseGridCpu(3, spec["size"], [np.float64] * 3, block_edge=8)
    n = spec["chunk_ids"].size
    g.insert_block(spec["chunk_ids"], np.ones((n, 512), np.uint8), [u_chunks, spec["f"], np.zeros((n, 512))])
    g.flush(["sright"] * 3)
    g.residual(0, 1, 2)
    r = g.prop(2)
    return float(np.sqrt((r * r).sum()) / np.sqrt((spec["f"] * spec["f"]).sum()))


def test_one_outer_iteration_matches_oracle(P, oracle):
    """max_outer = 1: defect (r = f), K FP32 red-black SOR sweeps of A e = r from e = 0,
    then u = 0 + e and its residual; u bit-exact against the oracle's sweeps."""
    specs = _small_grids(3, 11)
    K, w = 7, 1.37
    grids = [P.poisson_grid(s["size"], s["chunk_ids"], s["f"]) for s in specs]
    res = P.solve(grids, P.make_params(tol=1e-30, omega=w, first_sweeps=K, max_outer=1, use_graph=False))
    for s, g, r in zip(specs, grids, res):
        assert r["sweeps"] == K and r["outer"] == 1 and not r["converged"]
        u_gpu = g.prop(r["solution_prop"])
        n = s["chunk_ids"].size
        o = oracle.SparseGridCpu(3, s["size"], [np.float32, np.float32], block_edge=8)
        o.insert_block(s["chunk_ids"], np.ones((n, 512), np.uint8),
                       [np.zeros((n, 512), np.float32), s["f"].astype(np.float32)])
        o.flush(["sright", "sright"])
        for _ in range(K):
            o.rbsor_sweep(0, 1, w, 0)
            o.rbsor_sweep(0, 1, w, 1)
        e = o.prop(0).astype(np.float64)
        np.testing.assert_array_equal(u_gpu, 0.0 + e)
        rel = _oracle_residual(oracle, s, u_gpu)
        assert abs(rel - r["rel_residual"]) <= 1e-12 * rel


@pytest.mark.parametrize("mode", [C.POISSON_MIXED, C.POISSON_PLAIN_FP64])
@pytest.mark.parametrize("graph", [False, True])
def test_converges_to_1e_10(P, oracle, mode, graph):
    specs = _small_grids(6, 21 + mode)
    grids = [P.poisson_grid(s["size"], s["chunk_ids"], s["f"]) for s in specs]
    res = P.solve(grids, P.make_params(mode=mode, tol=1e-10, use_graph=graph))
    for s, g, r in zip(specs, grids, res):
        assert r["converged"], r
        assert r["rel_residual"] <= 1e-10
        rel = _oracle_residual(oracle, s, g.prop(r["solution_prop"]))
        assert rel <= 1.5e-10, (rel, r)


def test_mixed_against_all_fp64(P, oracle):
    """Error of the FP32+FP64 solution against the all-FP64 one.  Both have relative
    residual <= 1e-10; with kappa(A) = lambda_max / lambda_min <= 12 / 0.05 the relative
    2-norm difference of the solutions is bounded by 2 * kappa * 1e-10 = 4.8e-8."""
    specs = _small_grids(4, 31)
    gm = [P.poisson_grid(s["size"], s["chunk_ids"], s["f"]) for s in specs]
    gp = [P.poisson_grid(s["size"], s["chunk_ids"], s["f"]) for s in specs]
    rm = P.solve(gm, P.make_params(mode=C.POISSON_MIXED, tol=1e-10))
    rp = P.solve(gp, P.make_params(mode=C.POISSON_PLAIN_FP64, tol=1e-10))
    for a, b, ra, rb in zip(gm, gp, rm, rp):
        ua, ub = a.prop(ra["solution_prop"]), b.prop(rb["solution_prop"])
        err = np.linalg.norm(ua - ub) / np.linalg.norm(ub)
        assert err <= 4.8e-8, err


def test_alone_and_in_mix_identical(P):
    """Continuous batching: the iterates of a grid do not depend on its batch mates (each
    grid runs its own sweep counts inside the shared launches), so the solution is bitwise
    the same solved alone and admitted into a running batch of other grids."""
    import torch
    specs = _small_grids(7, 41)
    target = specs[3]
    g_alone = P.poisson_grid(target["size"], target["chunk_ids"], target["f"])
    r_alone = P.solve([g_alone], P.make_params(tol=1e-10))[0]
    u_alone = g_alone.prop(r_alone["solution_prop"])
    stream = torch.cuda.Stream()
    b = P.PoissonBatch(P.make_params(tol=1e-10), stream)
    grids = {}
    for i, s in enumerate(specs[:3]):
        grids[i] = P.poisson_grid(s["size"], s["chunk_ids"], s["f"], stream)
        b.add(grids[i], i)
    done = {}
    for step in range(200):
        if step == 2:  # admitted while the others are mid-solve
            for i, s in enumerate(specs[3:], start=3):
                grids[i] = P.poisson_grid(s["size"], s["chunk_ids"], s["f"], stream)
                b.add(grids[i], i)
        b.step()
        for tag, r in b.poll():
            done[tag] = r
        if len(done) == len(specs):
            break
    assert len(done) == len(specs) and all(r["converged"] for r in done.values())
    u_mix = grids[3].prop(done[3]["solution_prop"])
    assert done[3]["sweeps"] == r_alone["sweeps"]
    np.testing.assert_array_equal(u_mix, u_alone)
    b.close()


@pytest.mark.parametrize("waves,max_wgs", [(1, 0), (2, 7), (8, 0), (4, 33)])
def test_launch_shapes_identical(P, waves, max_wgs):
    """Waves per workgroup and looping waves (a workgroup cap) change only which wave
    sweeps which tile: solutions bitwise equal to the default launch shape."""
    specs = _small_grids(4, 51)
    ga = [P.poisson_grid(s["size"], s["chunk_ids"], s["f"]) for s in specs]
    gb = [P.poisson_grid(s["size"], s["chunk_ids"], s["f"]) for s in specs]
    ra = P.solve(ga, P.make_params(tol=1e-10))
    rb = P.solve(gb, P.make_params(tol=1e-10), tuning={C.TUNE_BATCH_WAVES: waves, C.TUNE_BATCH_MAX_WGS: max_wgs})
    for a, b, x, y in zip(ga, gb, ra, rb):
        assert x["sweeps"] == y["sweeps"] and y["converged"]
        np.testing.assert_array_equal(a.prop(x["solution_prop"]), b.prop(y["solution_prop"]))


@pytest.mark.parametrize("scale", [1.0, 4e-38, 2e-44])
@pytest.mark.parametrize("shape,sweeps,waves", [("points", 1, 4), ("points", 2, 1), ("points", 5, 4), ("block", 6, 2),
                                                ("one", 3, 4), ("diagonal", 4, 8)])
def test_fused_sweeps_match_oracle(P, oracle, shape, sweeps, waves, scale):
    """Both colours of a sweep in one pass, bit for bit the oracle's half sweeps: ragged point
    sets with padding-tagged points, a full block (every edge neighbour exists), a lone chunk,
    chunks that touch at edges and corners only (edge neighbours without a face neighbour);
    odd and even sweep counts (the last one writes e); right-hand sides whose quotients by 6
    are subnormal, ties among them (the true-division path)."""
    from openfpm_data_amd import SparseGridGpu
    import torch
    rng = np.random.default_rng(len(shape) + sweeps)
    n = 40
    if shape == "points":
        pts = W.shell_points(n, 6.0, 17.0)
        pts = pts[rng.random(len(pts)) < 0.9]
    else:
        lo = {"block": [(0, 0, 0), (24, 24, 24)], "one": [(8, 16, 8), (16, 24, 16)]}.get(shape)
        boxes = [lo] if lo else [((8 * i, 8 * j, 8 * k), (8 * i + 8, 8 * j + 8, 8 * k + 8))
                                 for i in range(4) for j in range(4) for k in range(4) if (i + j + k) % 2 == 0]
        pts = np.concatenate([np.stack(np.meshgrid(*[np.arange(a, b) for a, b in zip(*bx)], indexing="ij"), -1).reshape(-1, 3)
                              for bx in boxes])
    f = (rng.integers(-1000, 1000, len(pts)) * scale).astype(np.float32).astype(np.float64)
    z = np.zeros(len(pts))
    g = SparseGridGpu(3, (n,) * 3, P.POISSON_PROPS)
    g.insert_coords(pts.astype(np.int32), [z, z, f, z.astype(np.float32), z.astype(np.float32)])
    g.flush(["sright"] * 5)
    o = oracle.SparseGridCpu(3, (n,) * 3, [np.float32, np.float32], block_edge=8)
    o.insert_coords(pts.astype(np.int32), [z.astype(np.float32), f.astype(np.float32)])
    o.flush(["sright"] * 2)
    if shape == "points":
        g.tag_boundaries()
        o.tag_boundaries()
    torch.cuda.synchronize()
    r = P.solve([g], P.make_params(tol=1e-300, omega=1.37, first_sweeps=sweeps, max_outer=1, use_graph=sweeps % 2 == 0),
                tuning={C.TUNE_BATCH_WAVES: waves})[0]
    assert r["sweeps"] == sweeps
    for _ in range(sweeps):
        o.rbsor_sweep(0, 1, 1.37, 0)
        o.rbsor_sweep(0, 1, 1.37, 1)
    np.testing.assert_array_equal(g.masks(), o.masks())
    want = o.prop(0)
    assert want[want != 0].size > 0
    np.testing.assert_array_equal(g.prop(P.E).view(np.uint32), want.view(np.uint32))
    np.testing.assert_array_equal(g.prop(r["solution_prop"]), 0.0 + want.astype(np.float64))


def test_grids_without_fused_sweeps(P, oracle):
    """A background of e other than 0 (read where no point is) makes the step run half sweeps,
    for its batch mates as well: the mates' solutions keep their bits."""
    specs = _small_grids(2, 5, 48)
    alone = [P.poisson_grid(s["size"], s["chunk_ids"], s["f"]) for s in specs]
    ra = [P.solve([g], P.make_params(tol=1e-8))[0] for g in alone]
    mixed = [P.poisson_grid(s["size"], s["chunk_ids"], s["f"]) for s in specs]
    mixed[1].set_background_value(P.E, 0.5)
    rm = P.solve(mixed, P.make_params(tol=1e-8, max_outer=30))
    assert ra[0]["converged"] and rm[0]["converged"] and ra[0]["sweeps"] == rm[0]["sweeps"]
    np.testing.assert_array_equal(alone[0].prop(ra[0]["solution_prop"]), mixed[0].prop(rm[0]["solution_prop"]))


@pytest.mark.parametrize("sweeps", [1, 2, 5, 8])
def test_live_grid_changed_between_steps(P, sweeps):
    """Points removed (whole rows and a whole chunk), a chunk set that grows, shrinks again and
    a background of e that comes and goes, each between two steps of a live grid: the bits of
    half sweeps, which a mate with another background of e makes the step run."""
    import torch
    rng = np.random.default_rng(sweeps)
    n = 48
    boxes = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (1, 1, 1), (2, 1, 1), (4, 4, 4)]
    cells = np.stack(np.meshgrid(*[np.arange(8)] * 3, indexing="ij"), -1).reshape(-1, 3)
    pts = np.concatenate([cells + 8 * np.array(b) for b in boxes]).astype(np.int32)
    more = np.concatenate([cells + 8 * np.array(b) for b in [(2, 0, 0), (0, 1, 1), (5, 5, 5)]]).astype(np.int32)
    f, f2 = rng.uniform(-1, 1, len(pts)), rng.uniform(-1, 1, len(more))
    mate_spec = _small_grids(1, 5, 32)[0]

    def grid_values(half):
        from openfpm_data_amd import SparseGridGpu
        g = SparseGridGpu(3, (n,) * 3, P.POISSON_PROPS)
        put = lambda c, v: (g.insert_coords(c, [0 * v, 0 * v, v] + [np.zeros(len(c), np.float32)] * 2),  # noqa: E731
                            g.flush(["sright"] * 5))
        put(pts, f)
        b = P.PoissonBatch(P.make_params(tol=1e-300, omega=1.4, first_sweeps=sweeps, inner_target=0.3, max_outer=9,
                                         use_graph=sweeps % 2 == 0))
        b.add(g, 0)
        mate = P.poisson_grid(mate_spec["size"], mate_spec["chunk_ids"], mate_spec["f"])
        if half:
            mate.set_background_value(P.E, 0.5)
        b.add(mate, 1)
        seen = []
        for step in range(8):
            b.step()
            torch.cuda.synchronize()
            seen.append([g.prop(P.U), g.prop(P.U2), g.prop(P.E), g.prop(P.R)])
            if step == 1:  # rows and a chunk without a point
                gone = pts[(pts[:, 1] % 8 == 3) | (pts[:, 0] >= 32) | ((pts[:, 0] < 8) & (pts[:, 2] > 2))]
                g.remove_points(g.lin_id(gone))
            elif step == 3:
                put(more, f2)
            elif step == 4:
                g.set_background_value(P.E, 0.25)
            elif step == 5:
                g.set_background_value(P.E, 0.0)
            elif step == 6:
                keep = np.ascontiguousarray(g.chunk_ids()[::2])
                m = np.ascontiguousarray(g.masks()[::2])
                vals = [g.prop(p)[::2] for p in range(5)]
                C.check(g._lib.sg_set_chunks(g._h, len(keep), keep.ctypes.data, m.ctypes.data, C.SG_MEM_HOST))
                for p in range(5):
                    g.set_prop(p, vals[p])
            torch.cuda.synchronize()
        b.close()
        return seen

    for a, h in zip(grid_values(False), grid_values(True)):
        for x, y in zip(a, h):
            np.testing.assert_array_equal(x.view(np.uint8), y.view(np.uint8))


def test_waves_by_size_can_be_restored(P):
    """0 waves, the default (by the number of tiles), is accepted after another setting; the
    solutions do not depend on it."""
    import torch
    from openfpm_data_amd._capi import SgError
    spec = _small_grids(1, 7, 64)[0]
    out = []
    for settings in ((), (4,), (8, 0)):
        g = P.poisson_grid(spec["size"], spec["chunk_ids"], spec["f"])
        b = P.PoissonBatch(P.make_params(tol=1e-8), torch.cuda.current_stream())
        for w in settings:
            b.set_tuning(C.TUNE_BATCH_WAVES, w)
        for w in (-1, 3, 16):
            with pytest.raises(SgError):
                b.set_tuning(C.TUNE_BATCH_WAVES, w)
        b.add(g, 0)
        while b.live():
            b.step()
        res = b.poll()[0][1]
        b.close()
        out.append((res["sweeps"], g.prop(res["solution_prop"])))
    for sweeps, u in out[1:]:
        assert sweeps == out[0][0]
        np.testing.assert_array_equal(u, out[0][1])
