// sg_poisson.hip -- batched Poisson solves on 8^3-chunk sparse grids (gfx950).
//
// -lap(u) = f on the existing points of each grid, u = 0 outside (the background), with
// the 7-point operator A u = 6 u - sum of the 6 face neighbours.
//
// Precision form (SG_POISSON_MIXED): the state e and its right-hand side r are FP32 and
// swept with red-black SOR; FP64 is used only for the defect correction and the residual
// norms:   u' = u + e,   r = f - A u' (FP64),   ||r||, ||f|| (FP64),   e <- SOR sweeps of
// A e = (float) r from e = 0.  Plain form (SG_POISSON_PLAIN_FP64): red-black SOR sweeps of
// A u = f directly in FP64, residual checked between sweep blocks.
//
// Batching: every launch covers all live grids; workgroup waves take tiles of a (grid,
// chunk) work list (per-grid prefix sums of chunk counts, binary-searched per wave), so
// grids of uneven size share launches and small grids cost no launches of their own.
// An inner sweep sequence that comes again is captured in a hipGraph and replayed.
// Grids join and leave the batch between outer iterations (continuous batching).
//
// SOR relaxation: omega is estimated per grid from the residual reduction rho of each
// outer iteration (the first runs with omega0): the red-black ordered 7-point matrix is
// consistently ordered, so the SOR eigenvalue lambda and the Jacobi spectral radius mu
// satisfy (lambda + w - 1)^2 = lambda w^2 mu^2 (Young); mu from (rho, w), then
// omega_opt = 2 / (1 + sqrt(1 - mu^2)).
#include "sg_internal.hpp"

#include <algorithm>
#include <cmath>

namespace sg {
namespace {

struct PGrid {
    const int32_t *nn;    // NNStar table [n][8]
    const uint8_t *mask;  // [n+1][512]
    void *x;              // swept unknown (e: f32 mixed, u: f64 plain)
    const void *rhs;      // r (f32) or f (f64)
    const double *u_in;   // defect: current u
    double *u_out;        // defect: u + e
    const double *f;      // defect / residual: f
    float *e;             // defect: correction (may be null: treated as 0)
    float *r32;           // defect: FP32 residual written for the inner solve
    double omega;
    int64_t n;            // chunks
    int32_t nsweeps;      // sweeps of this grid in the current inner block
    // fused sweeps (mixed form): x's second buffer, the chunks' 18 neighbours, and whether they
    // are still to be set up
    float *x2;
    int32_t *nb;
    int32_t prep;
};

// A pointer of a grid descriptor in memory, read as one into global memory: as far as the
// compiler knows a plain one may point anywhere, and its accesses become flat ones, which
// also count as LDS accesses, wait for them, and take 64-bit addresses per lane.
template <typename T> __device__ __forceinline__ T *as_global(T *const &field)
{
    __attribute__((address_space(1))) T *g;
    __builtin_memcpy(&g, &field, sizeof(g));
    return (T *)g;
}

template <typename T> struct R8 {
    T v[8];
};

template <typename T> __device__ inline void ld8(R8<T> &r, const T *p)
{
    if constexpr (sizeof(T) == 4) {
        const float4 a = ((const float4 *)p)[0], b = ((const float4 *)p)[1];
        r.v[0] = a.x; r.v[1] = a.y; r.v[2] = a.z; r.v[3] = a.w;
        r.v[4] = b.x; r.v[5] = b.y; r.v[6] = b.z; r.v[7] = b.w;
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const double2 a = ((const double2 *)p)[i];
            r.v[2 * i] = a.x;
            r.v[2 * i + 1] = a.y;
        }
    }
}

template <typename T> __device__ inline void st8(T *p, const R8<T> &r)
{
    if constexpr (sizeof(T) == 4) {
        ((float4 *)p)[0] = make_float4(r.v[0], r.v[1], r.v[2], r.v[3]);
        ((float4 *)p)[1] = make_float4(r.v[4], r.v[5], r.v[6], r.v[7]);
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) ((double2 *)p)[i] = make_double2(r.v[2 * i], r.v[2 * i + 1]);
    }
}

__device__ inline void wave_sync_lds()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ghost half row of the +-y / +-z faces for lane (see sg_stencil.hip): source row in the
// neighbour chunk and destination row of the 10x10-row tile
__device__ inline int g_src_row(int lane)
{
    const int face = lane >> 4, idx = (lane >> 1) & 7;
    const int ry = idx * 8 + ((face == 0) ? 7 : 0);
    const int rz = ((face == 2) ? 56 : 0) + idx;
    return (face < 2) ? ry : rz;
}
__device__ inline int g_tile_row(int lane)
{
    const int face = lane >> 4, idx = (lane >> 1) & 7;
    const int ty = (idx + 1) * 10 + ((face == 0) ? 0 : 9);
    const int tz = ((face == 2) ? 0 : 90) + idx + 1;
    return (face < 2) ? ty : tz;
}

// Stage a property's own rows + face ghost rows in the tile, return own row and x ghosts.
template <typename T>
__device__ inline void stage(const T *arr, int64_t c, const int64_t (&nbp)[6], T *tile, int lane, R8<T> &own, T &xm,
                             T &xp)
{
    ld8(own, arr + c * 512 + lane * 8);
    const int face = lane >> 4;
    const int64_t nbc = (face == 0) ? nbp[2] : (face == 1) ? nbp[3] : (face == 2) ? nbp[4] : nbp[5];
    const T *src = arr + nbc * 512 + g_src_row(lane) * 8 + (lane & 1) * 4;
    T *dst = tile + g_tile_row(lane) * 8 + (lane & 1) * 4;
    if constexpr (sizeof(T) == 4) {
        *(float4 *)dst = *(const float4 *)src;
    } else {
        ((double2 *)dst)[0] = ((const double2 *)src)[0];
        ((double2 *)dst)[1] = ((const double2 *)src)[1];
    }
    xm = arr[nbp[0] * 512 + lane * 8 + 7];
    xp = arr[nbp[1] * 512 + lane * 8 + 0];
    const int y = lane & 7, z = lane >> 3;
    st8(tile + ((z + 1) * 10 + (y + 1)) * 8, own);
}

template <typename T>
__device__ inline void neighbour_rows(const T *tile, int lane, R8<T> &ym, R8<T> &yp, R8<T> &zm, R8<T> &zp)
{
    const int y = lane & 7, z = lane >> 3;
    ld8(ym, tile + ((z + 1) * 10 + y) * 8);
    ld8(yp, tile + ((z + 1) * 10 + y + 2) * 8);
    ld8(zm, tile + (z * 10 + y + 1) * 8);
    ld8(zp, tile + ((z + 2) * 10 + y + 1) * 8);
}

// One colour of a red-black SOR sweep on one tile (chunk c of grid g): x += w ((rhs + sum
// nb) / 6 - x) on the points of colour `color` ((x + y + z) & 1; chunk origins are
// multiples of 8, so the local coordinates decide).  zero_x: x is taken as 0 everywhere
// (first half sweep of an inner solve): points of the other colour are written 0.  Whole
// rows are stored; values of the other colour are written back unchanged (no other wave
// changes them in this half sweep).
template <typename T>
__device__ __forceinline__ void sweep_tile(const PGrid &g, int64_t c, T *tile, int lane, int color, int zero_x)
{
    T *x = (T *)as_global(g.x);
    const T *rhs = (const T *)as_global(g.rhs);
    const uint64_t mrow = *(const uint64_t *)(as_global(g.mask) + c * 512 + lane * 8);
    R8<T> b;
    ld8(b, rhs + c * 512 + lane * 8);
    R8<T> own, ym, yp, zm, zp;
    T xm = 0, xp = 0;
    if (zero_x) {
#pragma unroll
        for (int i = 0; i < 8; ++i) own.v[i] = ym.v[i] = yp.v[i] = zm.v[i] = zp.v[i] = (T)0;
    } else {
        int64_t nbp[6];
        const int32_t *row = as_global(g.nn) + c * 8;
#pragma unroll
        for (int k = 0; k < 6; ++k) nbp[k] = row[k];
        stage<T>(x, c, nbp, tile, lane, own, xm, xp);
        wave_sync_lds();
        neighbour_rows<T>(tile, lane, ym, yp, zm, zp);
    }
    const T wgt = (T)g.omega;
    const int par0 = ((lane & 7) + (lane >> 3)) & 1;  // parity of (y + z)
    R8<T> out;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint8_t cm = (uint8_t)(mrow >> (8 * i));
        const bool active = (cm & SG_EXIST) && !(cm & SG_PADDING);
        const bool mine = ((i + par0) & 1) == color;
        const T cur = own.v[i];
        const T l = (i == 0) ? xm : own.v[i - 1];
        const T r = (i == 7) ? xp : own.v[i + 1];
        T nbs = (T)0;
        nbs = nbs + (l + r);
        nbs = nbs + (ym.v[i] + yp.v[i]);
        nbs = nbs + (zm.v[i] + zp.v[i]);
        const T gs = (b.v[i] + nbs) / (T)6;
        const T nv = cur + wgt * (gs - cur);
        out.v[i] = (active && mine) ? nv : cur;
    }
    // rows with a point are written whole (both colours: the other colour keeps its
    // value): staged in the LDS tile, then written back as lane-contiguous 16-byte stores
    wave_sync_lds();  // every lane has read its neighbour rows
    st8(tile + lane * 8, out);
    wave_sync_lds();
    store_chunk_contig(x + c * 512, tile, mrow != 0 ? 1u : 0u, lane);
    // the next tile of this wave restages the LDS tile: finish reading it first
    wave_sync_lds();
}

// One colour of a red-black SOR sweep over the live grids.  Grids are ordered by
// decreasing sweep count, so the tiles of the grids still sweeping at sweep `sweep` are
// [0, act[sweep]); tile t belongs to grid tile_grid[t].  Wave v takes tiles v, v + V, ...
// (V = waves in the launch), so a launch of any size covers the active tiles.
template <typename T, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void rbsor_batch_kernel(const PGrid *__restrict__ grids,
                                                                const int64_t *__restrict__ prefix,
                                                                const int32_t *__restrict__ tile_grid,
                                                                const int64_t *__restrict__ act, int color,
                                                                int zero_x, int sweep)
{
    __shared__ __attribute__((aligned(16))) T tiles[WAVES][100 * 8];
    // uniform wave index: the tile's grid descriptor and neighbour-table row come by
    // scalar loads
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t nact = act[sweep];
    const int64_t nwaves = (int64_t)gridDim.x * WAVES;
    for (int64_t t = (int64_t)blockIdx.x * WAVES + w; t < nact; t += nwaves) {
        const int gi = tile_grid[t];
        sweep_tile<T>(grids[gi], t - prefix[gi], tiles[w], lane, color, zero_x);
    }
}

// ---- both colours of a sweep in one pass (FP32) ---------------------------------------
// A half sweep reads and writes every value of x for an update of half of them, so a sweep
// of two launches moves 26 B a slot.  Here a wave updates the first colour on its chunk and,
// a second time, on the ring of first-colour points of the six neighbour chunks' faces,
// which the chunk's second colour then uses: each value is computed from the same inputs by
// the same operations as in the neighbour's own wave, so the iterates keep their bits.  The
// ring's update needs a second layer of x, the ring's right-hand side and masks, and the
// values beside it in the 12 edge neighbours (those at nb[6 ..]).  x alternates between two
// buffers from sweep to sweep, the last sweep of a block writing the property (PGrid::x).
// Moved: 13 B a slot plus the ring, which other waves load as well (cache hits mostly), and
// half the launches.  The kernel is bound by instructions (about 400 vector ones a chunk,
// against 2 x 363 of two half sweeps); before the rows were kept split by colour, with a
// select for every operand, it had 680 and a sweep of 48 grids took 115 us.  Those 48 grids
// (58,600 chunks): 2 x 64 us a sweep in half sweeps, 66 us here; 152 chunks 2 x 4.8 -> 3.9 us.
// Measured and not kept (ms a solve of the 48, 10.0 then as it is): 1, 2 or 8 waves a workgroup
// 10.4, 10.3, 10.2; plain stores 10.4; contiguous tile ranges per XCD 10.1; groups of grids of
// 16,384 tiles one after the other, so that a group stays in the Infinity Cache, 11.6 (the
// launches' tails cost more than the misses).
constexpr int kNb = 20;  // entries per chunk: -x +x -y +y -z +z, xy, xz, yz edges, 2 unused
// LDS row of the 10 x 10 rows of a chunk and its ring: the 4 points of the first colour, the 4
// of the second, then x = -1 and x = 8 at 8 and 9.  Point j of a colour is at x = 2 j + s, s
// the row's parity for it; the rows above, below, before and behind have the other parity, so
// their points j of the other colour are its neighbours there: a row is updated from one
// 16-byte read of each of the four, with no selection.
constexpr int kFS = 12;

// neighbour tables and the second buffers' background chunks of the grids that joined the
// batch or whose chunk set changed (one wave per chunk): edge neighbour (a, b) is b's
// neighbour of a's neighbour, or where that is missing a's of b's; the background chunk where
// neither exists.  The second buffers' other chunks are first written by the sweeps.
__global__ __launch_bounds__(256) void fused_prep_kernel(const PGrid *__restrict__ grids,
                                                         const int64_t *__restrict__ prefix,
                                                         const int32_t *__restrict__ tile_grid, int64_t ntiles)
{
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t t = (int64_t)blockIdx.x * 4 + w;
    if (t >= ntiles) return;
    const int gi = tile_grid[t];
    const PGrid &g = grids[gi];
    if (!g.prep) return;
    const int64_t c = t - prefix[gi];
    if (c == 0) {
        const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
        float4 *b = (float4 *)(g.x2 + g.n * 512);
        b[lane] = zero;
        b[64 + lane] = zero;
    }
    if (lane >= kNb) return;
    int32_t v = (int32_t)g.n;
    if (lane < 6) {
        v = g.nn[c * 8 + lane];
    } else if (lane < 18) {
        const int k = (lane - 6) >> 2, q = (lane - 6) & 3;
        const int a = (k == 2 ? 2 : 0) + (q & 1), b = (k == 0 ? 2 : 4) + (q >> 1);
        const int32_t na = g.nn[c * 8 + a], nc = g.nn[c * 8 + b];
        if (na != v) v = g.nn[(int64_t)na * 8 + b];
        else if (nc != v) v = g.nn[(int64_t)nc * 8 + a];
    }
    g.nb[c * kNb + lane] = v;
}

__device__ __forceinline__ float sel(bool m, float a, float b) { return m ? a : b; }

// a / 6 correctly rounded: with y the rounded 1 / 6 (off by 2^-25 of it), a y is within one
// unit in the last place of a / 6, its remainder a - 6 q is exact, and one correction by it
// gives the rounded quotient (Markstein).  That needs a quotient in the normal range: *small
// is set where it is subnormal, and the caller divides.  Zeros, infinities and NaN are the
// fixup's.  5 instructions instead of 12.
__device__ __forceinline__ float div6(float a, bool *small)
{
    const float y = 1.0f / 6.0f;
    const float q = a * y;
    const float r = __builtin_fmaf(-6.0f, q, a);
    // class mask: negative and positive subnormals
    *small = *small || __builtin_amdgcn_classf(q, (1 << 4) | (1 << 7));
    return __builtin_amdgcn_div_fixupf(__builtin_fmaf(r, y, q), 6.0f, a);
}

// x + w ((b + nbs) / 6 - x) as sweep_tile computes it, where the point is active (mask m);
// EXACT: by true division
template <bool EXACT>
__device__ __forceinline__ float sor_value(float cur, float b, float px, float py, float pz, float wgt, uint32_t m,
                                           bool *small)
{
    float nbs = 0.0f;
    nbs = nbs + px;
    nbs = nbs + py;
    nbs = nbs + pz;
    const float a = b + nbs;
    const float gs = EXACT ? a / 6.0f : div6(a, small);
    const float x = cur + wgt * (gs - cur);
    return (m & (SG_EXIST | SG_PADDING)) == SG_EXIST ? x : cur;
}

// One colour on the lane's row: its points c[4], the other colour's o[4], the value end beside
// the row that points of parity s have (x = 8 for s, else x = -1), the neighbour rows' points
// of the other colour at p (LDS).  m: the row's masks.
template <bool EXACT>
__device__ __forceinline__ void sor_row(float (&c)[4], const float (&o)[4], const float (&b)[4], float end, bool s,
                                        const float *p, uint64_t m, float wgt, bool *small)
{
    const float4 ym = *(const float4 *)(p - kFS), yp = *(const float4 *)(p + kFS);
    const float4 zm = *(const float4 *)(p - 10 * kFS), zp = *(const float4 *)(p + 10 * kFS);
    const uint64_t ms = s ? m >> 8 : m;
    // l + r: o[j] on one side, o[j + 1] or o[j - 1] on the other
    const float x0 = o[0] + sel(s, o[1], end), x1 = o[1] + sel(s, o[2], o[0]);
    const float x2 = o[2] + sel(s, o[3], o[1]), x3 = o[3] + sel(s, end, o[2]);
    const uint32_t m0 = (uint32_t)ms, m1 = (uint32_t)(ms >> 32);
    c[0] = sor_value<EXACT>(c[0], b[0], x0, ym.x + yp.x, zm.x + zp.x, wgt, m0, small);
    c[1] = sor_value<EXACT>(c[1], b[1], x1, ym.y + yp.y, zm.y + zp.y, wgt, m0 >> 16, small);
    c[2] = sor_value<EXACT>(c[2], b[2], x2, ym.z + yp.z, zm.z + zp.z, wgt, m1, small);
    c[3] = sor_value<EXACT>(c[3], b[3], x3, ym.w + yp.w, zm.w + zp.w, wgt, m1 >> 16, small);
}

// the points of parity s (first) and the others of 8 values
__device__ __forceinline__ void split8(float (&a)[4], float (&b)[4], const R8<float> &v, bool s)
{
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        a[j] = sel(s, v.v[2 * j + 1], v.v[2 * j]);
        b[j] = sel(s, v.v[2 * j], v.v[2 * j + 1]);
    }
}

template <typename V> __device__ __forceinline__ V ld_at(const void *base, uint32_t byte)
{
    return *(const V *)((const char *)base + byte);
}

// per-lane values of one chunk for both colours
struct FusedIn {
    uint64_t mrow;                    // masks of the row
    float c0[4], c1[4], b0[4], b1[4]; // first and second colour of the row, their right-hand sides
    float xmm, xm, xp, xpp;           // x = -2, -1, 8, 9 of the row
    // the lane's half row of a y / z face of the ring: first colour, right-hand side, second
    // layer (beside the first colour), second colour, masks
    float2 r0, rb, rl, r1;
    uint32_t rm;
    float sb;     // right-hand side and mask of the ring's first-colour point beside the row
    uint32_t sm;
};

// Everything after the loads: EXACT divides truly; otherwise *small asks for that.  c0 and c1
// are updated.
template <bool EXACT>
__device__ __forceinline__ void fused_compute(FusedIn &in, float *tile, int lane, float wgt, bool *small)
{
    const int y = lane & 7, z = lane >> 3, face = lane >> 4, idx = (lane >> 1) & 7, half = lane & 1;
    const bool s = ((y + z) & 1) != 0;
    const int own = ((z + 1) * 10 + y + 1) * kFS, trow = g_tile_row(lane) * kFS;
    const bool yface = face < 2, rs = ((idx + ((face & 1) ? 0 : 1)) & 1) != 0;
    // the ring's half row
    float2 rn;
    {
        const int inner = (yface ? (idx + 1) * 10 + (face == 0 ? 1 : 8) : (face == 2 ? 10 : 80) + idx + 1) * kFS;
        const int d = (yface ? 10 : 1) * kFS, at = 4 + 2 * half;
        const float2 ip = *(const float2 *)(tile + inner + at);
        const float2 lo = *(const float2 *)(tile + trow - d + at), hi = *(const float2 *)(tile + trow + d + at);
        // the second colour's point beyond the half row that its parity has as a neighbour
        const float e = tile[trow + (rs ? (half ? 9 : 6) : (half ? 5 : 8))];
        const float n0 = in.rl.x + ip.x, n1 = in.rl.y + ip.y, a0 = lo.x + hi.x, a1 = lo.y + hi.y;
        rn.x = sor_value<EXACT>(in.r0.x, in.rb.x, in.r1.x + sel(rs, in.r1.y, e), sel(yface, n0, a0),
                                sel(yface, a0, n0), wgt, rs ? in.rm >> 8 : in.rm, small);
        rn.y = sor_value<EXACT>(in.r0.y, in.rb.y, in.r1.y + sel(rs, e, in.r1.x), sel(yface, n1, a1),
                                sel(yface, a1, n1), wgt, rs ? in.rm >> 24 : in.rm >> 16, small);
    }
    // the ring's point beside the row: x = -1 for rows of parity s, else x = 8
    const int sl = s ? 8 : 9;
    const float py = tile[own - kFS + sl] + tile[own + kFS + sl];
    const float pz = tile[own - 10 * kFS + sl] + tile[own + 10 * kFS + sl];
    const float xn = sor_value<EXACT>(sel(s, in.xm, in.xp), in.sb, sel(s, in.xmm, in.xpp) + sel(s, in.c1[0], in.c1[3]),
                                      py, pz, wgt, in.sm, small);
    // the row: first-colour points of parity s end beside x = 8, the others beside x = -1
    sor_row<EXACT>(in.c0, in.c1, in.b0, sel(s, in.xp, in.xm), s, tile + own + 4, in.mrow, wgt, small);
    wave_sync_lds();
    *(float4 *)(tile + own) = make_float4(in.c0[0], in.c0[1], in.c0[2], in.c0[3]);
    *(float2 *)(tile + trow + 2 * half) = rn;
    wave_sync_lds();
    // second-colour points have the other parity: they end beside the updated ring point
    sor_row<EXACT>(in.c1, in.c0, in.b1, xn, !s, tile + own, in.mrow, wgt, small);
}

// both colours on chunk c of grid g (fewer than 2^21 chunks: 32-bit byte offsets): src -> dst,
// the rows with a point and those of `every`
__device__ __forceinline__ void fused_tile(const PGrid &g, uint32_t c, float *tile, int lane, int zero_x,
                                           const float *src, float *dst, uint64_t every)
{
    const int32_t *nb = as_global(g.nb) + (size_t)c * kNb;
    const float *rhs = (const float *)as_global(g.rhs);
    const uint8_t *mask = as_global(g.mask);
    const int y = lane & 7, z = lane >> 3, face = lane >> 4, idx = (lane >> 1) & 7, half = lane & 1;
    const bool s = ((y + z) & 1) != 0, rs = ((idx + ((face & 1) ? 0 : 1)) & 1) != 0;
    const int own = ((z + 1) * 10 + y + 1) * kFS, trow = g_tile_row(lane) * kFS;
    // source rows of the ring's half row in the neighbour: first and second layer
    const int row1 = g_src_row(lane);
    const int row2 = face < 2 ? idx * 8 + (face == 0 ? 6 : 1) : (face == 2 ? 48 : 8) + idx;
    const uint32_t n0 = (uint32_t)nb[0], n1 = (uint32_t)nb[1];
    const uint32_t nf = (uint32_t)(face < 2 ? (face == 0 ? nb[2] : nb[3]) : (face == 2 ? nb[4] : nb[5]));
    const uint32_t at = c * 2048u + (uint32_t)lane * 32u, atf = nf * 2048u + (uint32_t)half * 16u;
    // the ring's first-colour point beside the row
    const uint32_t side = (s ? n0 : n1) * 512u + (uint32_t)lane * 8u + (s ? 7u : 0u);

    FusedIn in;
    in.mrow = ld_at<uint64_t>(mask, c * 512u + (uint32_t)lane * 8u);
    R8<float> b, u;
    ld8(b, (const float *)((const char *)rhs + at));
    const float4 bh = ld_at<float4>(rhs, atf + (uint32_t)row1 * 32u);
    in.rm = ld_at<uint32_t>(mask, nf * 512u + (uint32_t)row1 * 8u + (uint32_t)half * 4u);
    in.sb = ld_at<float>(rhs, side * 4u);
    in.sm = mask[side];
    float4 h1 = make_float4(0.f, 0.f, 0.f, 0.f), h2 = h1, ye = h1;
    float2 xm = make_float2(0.f, 0.f), xp = xm;
    float xe = 0.f;
    // edge values: lanes (e, i) -> value i of xy / xz edge e, one each; lanes 0 - 7 -> half rows
    // of the 4 yz edges
    const int ek = lane >> 5, es = (lane >> 4) & 1, ex = (lane >> 3) & 1, ei = lane & 7;
    const int erow = ek == 0 ? ei * 8 + (es ? 0 : 7) : (es ? 0 : 56) + ei;
    const int etile = (ek == 0 ? (ei + 1) * 10 + (es ? 9 : 0) : (es ? 90 : 0) + ei + 1) * kFS;
    const int ys = (lane >> 1) & 1, zs = (lane >> 2) & 1;
    if (zero_x) {
#pragma unroll
        for (int i = 0; i < 8; ++i) u.v[i] = 0.f;
    } else {
        ld8(u, (const float *)((const char *)src + at));
        h1 = ld_at<float4>(src, atf + (uint32_t)row1 * 32u);
        h2 = ld_at<float4>(src, atf + (uint32_t)row2 * 32u);
        xm = ld_at<float2>(src, n0 * 2048u + (uint32_t)lane * 32u + 24u);
        xp = ld_at<float2>(src, n1 * 2048u + (uint32_t)lane * 32u);
        const uint32_t ne = (uint32_t)(ek == 0 ? (es ? (ex ? nb[9] : nb[8]) : (ex ? nb[7] : nb[6]))
                                               : (es ? (ex ? nb[13] : nb[12]) : (ex ? nb[11] : nb[10])));
        xe = ld_at<float>(src, ne * 2048u + (uint32_t)(erow * 8 + (ex ? 0 : 7)) * 4u);
        if (lane < 8) {
            const uint32_t ny = (uint32_t)(zs ? (ys ? nb[17] : nb[16]) : (ys ? nb[15] : nb[14]));
            ye = ld_at<float4>(src, ny * 2048u + (uint32_t)((zs ? 0 : 56) + (ys ? 0 : 7)) * 32u + (uint32_t)half * 16u);
        }
    }
    split8(in.c0, in.c1, u, s);
    split8(in.b0, in.b1, b, s);
    in.xmm = xm.x;
    in.xm = xm.y;
    in.xp = xp.x;
    in.xpp = xp.y;
    in.r0 = make_float2(sel(rs, h1.y, h1.x), sel(rs, h1.w, h1.z));
    in.r1 = make_float2(sel(rs, h1.x, h1.y), sel(rs, h1.z, h1.w));
    in.rl = make_float2(sel(rs, h2.y, h2.x), sel(rs, h2.w, h2.z));
    in.rb = make_float2(sel(rs, bh.y, bh.x), sel(rs, bh.w, bh.z));
    // the first colour's update reads second-colour points only
    *(float4 *)(tile + own + 4) = make_float4(in.c1[0], in.c1[1], in.c1[2], in.c1[3]);
    *(float2 *)(tile + own + 8) = make_float2(in.xm, in.xp);
    *(float2 *)(tile + trow + 4 + 2 * half) = in.r1;
    tile[etile + 8 + ex] = xe;
    if (lane < 8) {
        const bool cs = ys != zs;  // parity of the edge row (y and z are -1 or 8)
        *(float2 *)(tile + ((zs ? 90 : 0) + (ys ? 9 : 0)) * kFS + 4 + 2 * half) =
            make_float2(sel(cs, ye.x, ye.y), sel(cs, ye.z, ye.w));
    }
    wave_sync_lds();

    const float wgt = (float)g.omega;
    bool small = false;
    fused_compute<false>(in, tile, lane, wgt, &small);
    if (__ballot(small) != 0) {
        // subnormal quotients somewhere in the chunk: again with true divisions.  The LDS rows'
        // second-colour points are as they were, the first colour's are rewritten.
        R8<float> again;
#pragma unroll
        for (int i = 0; i < 8; ++i) again.v[i] = 0.f;
        if (!zero_x) ld8(again, (const float *)((const char *)src + at));
        split8(in.c0, in.c1, again, s);
        wave_sync_lds();
        fused_compute<true>(in, tile, lane, wgt, &small);
    }
    const uint64_t rows = __ballot(in.mrow != 0) | every;
    wave_sync_lds();
    // back in row order, and out as lane-contiguous 16-byte stores
    *(float4 *)(tile + lane * 8) = make_float4(sel(s, in.c1[0], in.c0[0]), sel(s, in.c0[0], in.c1[0]),
                                               sel(s, in.c1[1], in.c0[1]), sel(s, in.c0[1], in.c1[1]));
    *(float4 *)(tile + lane * 8 + 4) = make_float4(sel(s, in.c1[2], in.c0[2]), sel(s, in.c0[2], in.c1[2]),
                                                   sel(s, in.c1[3], in.c0[3]), sel(s, in.c0[3], in.c1[3]));
    wave_sync_lds();
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int v = k * 64 + lane;
        if ((rows >> (v >> 1)) & 1ull) copy16_nt((float *)((char *)dst + c * 2048u + (uint32_t)v * 16u), tile + v * 4);
    }
    // the next tile of this wave restages the LDS tile: finish reading it first
    wave_sync_lds();
}

// Sweep `sweep` of the live grids, both colours (work list as for rbsor_batch_kernel).  A tile
// per wave, or with LOOP as many as the launch's size needs: without the loop the per-lane
// offsets are not kept across it, 75 registers instead of 104, which allow 6 waves a SIMD
// instead of 4.
template <int WAVES, bool LOOP>
__global__ __launch_bounds__(64 * WAVES) void rbsor_fused_kernel(const PGrid *__restrict__ grids,
                                                                const int64_t *__restrict__ prefix,
                                                                const int32_t *__restrict__ tile_grid,
                                                                const int64_t *__restrict__ act, int zero_x, int sweep)
{
    __shared__ __attribute__((aligned(16))) float tiles[WAVES][100 * kFS];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t nact = act[sweep];
    auto tile = [&](int64_t t) __attribute__((always_inline)) {
        const int gi = tile_grid[t];
        const PGrid &g = grids[gi];
        // the block's last sweep writes x.  The rows without a point hold zeros in x, but in x2
        // whatever they held when they last had one: a block's first sweep into x2 writes all rows
        const bool to2 = ((g.nsweeps - 1 - sweep) & 1) != 0;
        float *x = (float *)as_global(g.x), *x2 = as_global(g.x2);
        fused_tile(g, (uint32_t)(t - prefix[gi]), tiles[w], lane, zero_x, to2 ? x : x2, to2 ? x2 : x,
                   to2 && sweep < 2 ? ~0ull : 0ull);
    };
    int64_t t = (int64_t)blockIdx.x * WAVES + w;
    if constexpr (LOOP) {
        for (; t < nact; t += (int64_t)gridDim.x * WAVES) tile(t);
    } else if (t < nact) {
        tile(t);
    }
}

// tile -> grid map of a work list
__global__ __launch_bounds__(256) void tile_grid_kernel(const int64_t *__restrict__ prefix, int32_t *__restrict__ tg)
{
    const int gi = blockIdx.x;
    for (int64_t t = prefix[gi] + threadIdx.x; t < prefix[gi + 1]; t += 256) tg[t] = gi;
}

// Defect correction + residual, FP64: u_out = u_in + e, r = f - A u_out, r32 = (float) r;
// per-tile partial sums of r^2 and f^2 over the existing points (reduced per grid in a
// fixed order afterwards, so the norms are deterministic).  e == nullptr: e = 0,
// u_out == nullptr: residual only.
__global__ __launch_bounds__(256) void defect_batch_kernel(const PGrid *__restrict__ grids,
                                                           const int64_t *__restrict__ prefix,
                                                           const int32_t *__restrict__ tile_grid, int64_t ntiles,
                                                           double *__restrict__ partial)
{
    __shared__ __attribute__((aligned(16))) double tiles[4][100 * 8];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t t = (int64_t)blockIdx.x * 4 + w;
    if (t >= ntiles) return;
    const int gi = tile_grid[t];
    const PGrid &gd = grids[gi];
    struct {
        const int32_t *nn;
        const uint8_t *mask;
        const double *u_in, *f;
        double *u_out;
        const float *e;
        float *r32;
    } g = {as_global(gd.nn), as_global(gd.mask), as_global(gd.u_in), as_global(gd.f),
           as_global(gd.u_out), as_global(gd.e), as_global(gd.r32)};
    const int64_t c = t - prefix[gi];
    int64_t nbp[6];
    const int32_t *row = g.nn + c * 8;
#pragma unroll
    for (int k = 0; k < 6; ++k) nbp[k] = row[k];
    const uint64_t mrow = *(const uint64_t *)(g.mask + c * 512 + lane * 8);
    R8<double> u, fr;
    double uxm, uxp;
    double *tile = tiles[w];
    // stage u (+ e) : u' = u + e for own rows and ghosts
    {
        ld8(u, g.u_in + c * 512 + lane * 8);
        const int face = lane >> 4;
        const int64_t nbc = (face == 0) ? nbp[2] : (face == 1) ? nbp[3] : (face == 2) ? nbp[4] : nbp[5];
        const int64_t goff = nbc * 512 + g_src_row(lane) * 8 + (lane & 1) * 4;
        double gh[4];
        const double2 a = ((const double2 *)(g.u_in + goff))[0], bb = ((const double2 *)(g.u_in + goff))[1];
        gh[0] = a.x; gh[1] = a.y; gh[2] = bb.x; gh[3] = bb.y;
        uxm = g.u_in[nbp[0] * 512 + lane * 8 + 7];
        uxp = g.u_in[nbp[1] * 512 + lane * 8 + 0];
        if (g.e) {
            R8<float> e;
            ld8(e, g.e + c * 512 + lane * 8);
#pragma unroll
            for (int i = 0; i < 8; ++i) u.v[i] = u.v[i] + (double)e.v[i];
            const float4 eg = *(const float4 *)(g.e + goff);
            gh[0] = gh[0] + (double)eg.x; gh[1] = gh[1] + (double)eg.y;
            gh[2] = gh[2] + (double)eg.z; gh[3] = gh[3] + (double)eg.w;
            uxm = uxm + (double)g.e[nbp[0] * 512 + lane * 8 + 7];
            uxp = uxp + (double)g.e[nbp[1] * 512 + lane * 8 + 0];
        }
        double *dst = tile + g_tile_row(lane) * 8 + (lane & 1) * 4;
        ((double2 *)dst)[0] = make_double2(gh[0], gh[1]);
        ((double2 *)dst)[1] = make_double2(gh[2], gh[3]);
        const int y = lane & 7, z = lane >> 3;
        st8(tile + ((z + 1) * 10 + (y + 1)) * 8, u);
    }
    ld8(fr, g.f + c * 512 + lane * 8);
    wave_sync_lds();
    R8<double> ym, yp, zm, zp;
    neighbour_rows<double>(tile, lane, ym, yp, zm, zp);
    double s_r = 0.0, s_f = 0.0;
    R8<float> r32;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint8_t cm = (uint8_t)(mrow >> (8 * i));
        const bool active = (cm & SG_EXIST) && !(cm & SG_PADDING);
        const double l = (i == 0) ? uxm : u.v[i - 1];
        const double rr = (i == 7) ? uxp : u.v[i + 1];
        double acc = 6.0 * u.v[i];
        acc = acc - (l + rr);
        acc = acc - (ym.v[i] + yp.v[i]);
        acc = acc - (zm.v[i] + zp.v[i]);
        const double res = fr.v[i] - acc;
        r32.v[i] = active ? (float)res : 0.0f;
        if (active) {
            s_r += res * res;
            s_f += fr.v[i] * fr.v[i];
        }
    }
    if (mrow != 0) {
        if (g.u_out) st8(g.u_out + c * 512 + lane * 8, u);
        if (g.r32) st8(g.r32 + c * 512 + lane * 8, r32);
    }
    // wave reduction (fixed shape)
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        s_r += __shfl_down(s_r, o, 64);
        s_f += __shfl_down(s_f, o, 64);
    }
    if (lane == 0) {
        partial[2 * t] = s_r;
        partial[2 * t + 1] = s_f;
    }
}

// per grid: sum of its tiles' partials in a fixed order (strided lanes + fixed tree)
__global__ __launch_bounds__(256) void norm_reduce_kernel(const double *__restrict__ partial,
                                                          const int64_t *__restrict__ prefix, int ng,
                                                          double *__restrict__ norms)
{
    __shared__ double sr[256], sf[256];
    const int gi = blockIdx.x;
    if (gi >= ng) return;
    double a = 0.0, b = 0.0;
    for (int64_t t = prefix[gi] + threadIdx.x; t < prefix[gi + 1]; t += 256) {
        a += partial[2 * t];
        b += partial[2 * t + 1];
    }
    sr[threadIdx.x] = a;
    sf[threadIdx.x] = b;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            sr[threadIdx.x] += sr[threadIdx.x + s];
            sf[threadIdx.x] += sf[threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        norms[2 * gi] = sr[0];
        norms[2 * gi + 1] = sf[0];
    }
}

}  // namespace
}  // namespace sg

struct sg_batch {
    sg_poisson_params p;
    hipStream_t stream = nullptr;
    bool own_stream = false;  // created here when the caller passed none (graphs need one)
    struct Entry {
        sg_grid *g;
        int64_t tag;
        int cur_u;  // property holding the current u (mixed: u_prop or u2_prop)
        int outer = 0;
        int sweeps = 0;
        double omega = 0.0;
        double norm_f = -1.0;
        double last_rel = -1.0;
        double rel = 1.0;
        int inner = 0;  // inner sweeps for the next outer iteration
        double tol = 0.0;
        // fused sweeps: second x buffer and neighbour table (from the batch's pool; null: the
        // grid cannot take them) for the chunk set of that count, still to be set up
        float *x2 = nullptr;
        int32_t *nb = nullptr;
        bool prep = false;
        uint64_t chunks_gen = 0;
    };
    std::vector<Entry> live;
    std::vector<std::pair<int64_t, sg_poisson_result>> done;
    // device work list (rebuilt when the live set changes)
    sg::DevicePool pool;
    sg::DevBuf d_list, d_partial, d_tg;
    // the work list's parts in d_list
    sg::PGrid *d_grids = nullptr;
    int64_t *d_prefix = nullptr, *d_act = nullptr;
    bool dirty = true;
    std::vector<int64_t> h_prefix, h_act;
    // pinned staging of the work lists (one for the defect's, one for the sweeps', so that a
    // list is rewritten only after a wait for the norms that follow its copy) and of the norms,
    // which their kernel writes there
    sg::PinnedBlock h_list[2], h_norms;
    // launch shape of the sweep kernel: waves per workgroup (1, 2, 4, 8; 0: by the number of
    // tiles) and a cap on the workgroups of one launch (0: one tile per wave); set by
    // sg_batch_set_tuning
    int waves = 0;
    int64_t max_wgs = 0;
    // graph of the inner sweep sequence for a live set and sweep count, and the last sequence
    // that was launched without one
    hipGraphExec_t graph = nullptr;
    int graph_sweeps = -1, last_sweeps = -1;
    uint64_t graph_version = 0, last_version = 0, version = 0;
    ~sg_batch()
    {
        if (graph) (void)hipGraphExecDestroy(graph);
        for (sg::PinnedBlock *h : {&h_list[0], &h_list[1], &h_norms}) sg::pinned_give(*h);
        pool.release();
    }
};

namespace {

using namespace sg;

int ensure_pinned(PinnedBlock &h, size_t bytes)
{
    if (h.bytes >= bytes) return SG_OK;
    pinned_give(h);
    return pinned_take(h, bytes + bytes / 2) ? SG_OK : fail(SG_E_OOM, "pinned host allocation failed");
}

// Device work list of the live grids in the order `order` (indices into live): grid
// descriptors, prefix sums of chunk counts, the tile -> grid map and, for the sweeps, the
// active tile count per sweep index (order must then be by decreasing inner count).
int upload_worklist(sg_batch *b, bool defect_view, const std::vector<int> &order)
{
    const int ng = (int)order.size();
    int max_inner = 1;
    for (const auto &en : b->live) max_inner = std::max(max_inner, en.inner);
    // one pinned block and one copy: descriptors | prefix sums | active tiles per sweep
    const size_t at_prefix = sizeof(PGrid) * (size_t)std::max(ng, 1), at_act = at_prefix + sizeof(int64_t) * (ng + 1);
    const size_t bytes = at_act + sizeof(int64_t) * (size_t)max_inner;
    PinnedBlock &hl = b->h_list[defect_view ? 0 : 1];
    const void *const had = b->d_list.p;
    int rc;
    if ((rc = ensure_pinned(hl, bytes)) || (rc = ensure(b->pool, b->d_list, bytes))) return rc;
    if (b->d_list.p != had) ++b->version;  // a captured sequence reads the old list
    PGrid *gd = (PGrid *)hl.p;
    b->h_prefix.assign(ng + 1, 0);
    const bool mixed = b->p.mode == SG_POISSON_MIXED;
    for (int i = 0; i < ng; ++i) {
        sg_batch::Entry &en = b->live[order[i]];
        sg_grid *g = en.g;
        PGrid &d = gd[i];
        d.nn = g->d_nn[SG_NN_STAR];
        d.mask = g->d_mask;
        d.n = g->nchunks;
        d.omega = en.omega;
        d.nsweeps = en.inner;
        d.f = (const double *)g->d_prop[b->p.f_prop];
        d.x2 = en.x2;
        d.nb = en.nb;
        d.prep = en.prep ? 1 : 0;
        if (mixed) {
            d.x = g->d_prop[b->p.e_prop];
            d.rhs = g->d_prop[b->p.r_prop];
            d.u_in = (const double *)g->d_prop[en.cur_u];
            const int other = (en.cur_u == b->p.u_prop) ? b->p.u2_prop : b->p.u_prop;
            d.u_out = defect_view ? (double *)g->d_prop[other] : nullptr;
            // the first defect of a grid takes u as given (e may hold an earlier solve's state)
            d.e = (defect_view && en.outer == 0) ? nullptr : (float *)g->d_prop[b->p.e_prop];
            d.r32 = (float *)g->d_prop[b->p.r_prop];
        } else {
            d.x = g->d_prop[b->p.u_prop];
            d.rhs = g->d_prop[b->p.f_prop];
            d.u_in = (const double *)g->d_prop[b->p.u_prop];
            d.u_out = nullptr;
            d.e = nullptr;
            d.r32 = nullptr;
        }
        b->h_prefix[i + 1] = b->h_prefix[i] + g->nchunks;
    }
    // act[s] = tiles of the grids with more than s sweeps (a prefix of the ordered list)
    b->h_act.assign(max_inner, 0);
    if (!defect_view) {
        int k = ng;
        for (int sw = 0; sw < max_inner; ++sw) {
            while (k > 0 && gd[k - 1].nsweeps <= sw) --k;
            b->h_act[sw] = b->h_prefix[k];
        }
    }
    const int64_t nt = b->h_prefix[ng];
    if ((rc = ensure(b->pool, b->d_partial, sizeof(double) * 2 * std::max<int64_t>(nt, 1))) ||
        (rc = ensure_pinned(b->h_norms, sizeof(double) * 2 * std::max(ng, 1))) ||
        (rc = ensure(b->pool, b->d_tg, sizeof(int32_t) * std::max<int64_t>(nt, 1))))
        return rc;
    memcpy((char *)hl.p + at_prefix, b->h_prefix.data(), sizeof(int64_t) * (ng + 1));
    memcpy((char *)hl.p + at_act, b->h_act.data(), sizeof(int64_t) * b->h_act.size());
    b->d_grids = (PGrid *)b->d_list.p;
    b->d_prefix = (int64_t *)((char *)b->d_list.p + at_prefix);
    b->d_act = (int64_t *)((char *)b->d_list.p + at_act);
    SG_HIP(hipMemcpyAsync(b->d_list.p, hl.p, bytes, hipMemcpyHostToDevice, b->stream));
    if (ng > 0) {
        hipLaunchKernelGGL(tile_grid_kernel, dim3((unsigned)ng), dim3(256), 0, b->stream, (const int64_t *)b->d_prefix,
                           (int32_t *)b->d_tg.p);
        SG_HIP(hipGetLastError());
    }
    return SG_OK;
}

// waves per workgroup of the sweeps: 4 (neighbour chunks share a CU's cache: the 48 grids above
// 10.0 ms, 10.4 ms with 1), or 1 while the tiles are fewer than would give every CU 4 waves
// (152 tiles: 4.3 us a sweep with 4 waves on 38 CUs, 3.9 us with 1 on 152)
int sweep_waves(const sg_batch *b, int64_t nt)
{
    if (b->waves > 0) return b->waves;
    return nt <= 1024 ? 1 : 4;
}

template <typename T, int W> int launch_sweep_kernel(sg_batch *b, unsigned nblk, int color, int zx, int s)
{
    hipLaunchKernelGGL((rbsor_batch_kernel<T, W>), dim3(nblk), dim3(64 * W), 0, b->stream,
                       (const PGrid *)b->d_grids, (const int64_t *)b->d_prefix, (const int32_t *)b->d_tg.p,
                       (const int64_t *)b->d_act, color, zx, s);
    SG_HIP(hipGetLastError());
    return SG_OK;
}

template <typename T> int launch_sweep(sg_batch *b, int waves, unsigned nblk, int color, int zx, int s)
{
    switch (waves) {
    case 1: return launch_sweep_kernel<T, 1>(b, nblk, color, zx, s);
    case 2: return launch_sweep_kernel<T, 2>(b, nblk, color, zx, s);
    case 8: return launch_sweep_kernel<T, 8>(b, nblk, color, zx, s);
    default: return launch_sweep_kernel<T, 4>(b, nblk, color, zx, s);
    }
}

// loop: fewer workgroups than tiles
template <int W> int launch_fused_kernel(sg_batch *b, unsigned nblk, bool loop, int zx, int s)
{
    if (loop)
        hipLaunchKernelGGL((rbsor_fused_kernel<W, true>), dim3(nblk), dim3(64 * W), 0, b->stream,
                           (const PGrid *)b->d_grids, (const int64_t *)b->d_prefix, (const int32_t *)b->d_tg.p,
                           (const int64_t *)b->d_act, zx, s);
    else
        hipLaunchKernelGGL((rbsor_fused_kernel<W, false>), dim3(nblk), dim3(64 * W), 0, b->stream,
                           (const PGrid *)b->d_grids, (const int64_t *)b->d_prefix, (const int32_t *)b->d_tg.p,
                           (const int64_t *)b->d_act, zx, s);
    SG_HIP(hipGetLastError());
    return SG_OK;
}

// every live grid can take fused sweeps (a grid that cannot makes the step run half sweeps
// for all: e ends in its property either way)
bool fused_ok(const sg_batch *b, bool first_zero)
{
    if (b->p.mode != SG_POISSON_MIXED || !first_zero) return false;
    for (const auto &en : b->live)
        if (!en.x2) return false;
    return true;
}

int launch_sweeps(sg_batch *b, int sweeps, bool first_zero)
{
    const int64_t nt = b->h_act.empty() ? 0 : b->h_act[0];
    if (nt == 0) return SG_OK;
    const int waves = sweep_waves(b, nt);
    int64_t nblk = (nt + waves - 1) / waves;
    if (b->max_wgs > 0) nblk = std::min(nblk, b->max_wgs);
    const bool mixed = b->p.mode == SG_POISSON_MIXED;
    if (fused_ok(b, first_zero)) {
        const bool loop = nblk * waves < nt;
        for (int s = 0; s < sweeps; ++s) {
            const int zx = s == 0 ? 1 : 0;
            int rc;
            switch (waves) {
            case 1: rc = launch_fused_kernel<1>(b, (unsigned)nblk, loop, zx, s); break;
            case 2: rc = launch_fused_kernel<2>(b, (unsigned)nblk, loop, zx, s); break;
            case 8: rc = launch_fused_kernel<8>(b, (unsigned)nblk, loop, zx, s); break;
            default: rc = launch_fused_kernel<4>(b, (unsigned)nblk, loop, zx, s); break;
            }
            if (rc) return rc;
        }
        return SG_OK;
    }
    for (int s = 0; s < sweeps; ++s) {
        for (int color = 0; color < 2; ++color) {
            const int zx = (first_zero && s == 0 && color == 0) ? 1 : 0;
            int rc = mixed ? launch_sweep<float>(b, waves, (unsigned)nblk, color, zx, s)
                           : launch_sweep<double>(b, waves, (unsigned)nblk, color, zx, s);
            if (rc) return rc;
        }
    }
    return SG_OK;
}

// run `sweeps` inner sweeps for the whole live set, through a cached hipGraph when asked: the
// sequence is captured when the same one comes a second time (capturing and instantiating 40
// launches takes the host longer than queuing them while the first already run)
int run_sweeps(sg_batch *b, int sweeps, bool first_zero)
{
    const bool have = b->graph && b->graph_sweeps == sweeps && b->graph_version == b->version;
    const bool again = b->last_sweeps == sweeps && b->last_version == b->version;
    if (!b->p.use_graph || (!have && !again)) {
        b->last_sweeps = sweeps;
        b->last_version = b->version;
        return launch_sweeps(b, sweeps, first_zero);
    }
    if (!b->graph || b->graph_sweeps != sweeps || b->graph_version != b->version) {
        if (b->graph) {
            SG_HIP(hipGraphExecDestroy(b->graph));
            b->graph = nullptr;
        }
        hipGraph_t gr;
        SG_HIP(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
        int rc = launch_sweeps(b, sweeps, first_zero);
        hipError_t e2 = hipStreamEndCapture(b->stream, &gr);
        if (rc) return rc;
        if (e2 != hipSuccess) return fail(SG_E_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e2));
        SG_HIP(hipGraphInstantiate(&b->graph, gr, nullptr, nullptr, 0));
        SG_HIP(hipGraphDestroy(gr));
        b->graph_sweeps = sweeps;
        b->graph_version = b->version;
    }
    SG_HIP(hipGraphLaunch(b->graph, b->stream));
    return SG_OK;
}

// defect (mixed) or residual (plain) over the live set; per-grid norms to the host
int defect_and_norms(sg_batch *b, std::vector<double> &norms, bool defect_view)
{
    const int ng = (int)b->live.size();
    std::vector<int> order(ng);
    for (int i = 0; i < ng; ++i) order[i] = i;
    int rc = upload_worklist(b, defect_view, order);
    if (rc) return rc;
    const int64_t nt = b->h_prefix[ng];
    norms.assign(2 * ng, 0.0);
    bool prep = false;
    for (const auto &en : b->live) prep = prep || en.prep;
    if (prep) {
        hipLaunchKernelGGL(fused_prep_kernel, dim3((unsigned)((nt + 3) / 4)), dim3(256), 0, b->stream,
                           (const PGrid *)b->d_grids, (const int64_t *)b->d_prefix, (const int32_t *)b->d_tg.p, nt);
        SG_HIP(hipGetLastError());
        for (auto &en : b->live) en.prep = false;
    }
    if (nt > 0) {
        hipLaunchKernelGGL(defect_batch_kernel, dim3((unsigned)((nt + 3) / 4)), dim3(256), 0, b->stream,
                           (const PGrid *)b->d_grids, (const int64_t *)b->d_prefix, (const int32_t *)b->d_tg.p,
                           nt, (double *)b->d_partial.p);
        SG_HIP(hipGetLastError());
        hipLaunchKernelGGL(norm_reduce_kernel, dim3((unsigned)ng), dim3(256), 0, b->stream,
                           (const double *)b->d_partial.p, (const int64_t *)b->d_prefix, ng, (double *)b->h_norms.p);
        SG_HIP(hipGetLastError());
        SG_HIP(hipStreamSynchronize(b->stream));
        memcpy(norms.data(), b->h_norms.p, sizeof(double) * 2 * ng);
    }
    return SG_OK;
}

// inner sweeps needed for a residual reduction `target` with SOR rate rho
int sweeps_for(double rho, double target, int lo, int hi)
{
    if (!(rho > 0.0) || rho >= 1.0) return hi;
    int k = (int)std::ceil(std::log(target) / std::log(rho));
    return std::max(lo, std::min(hi, k));
}

// Young's relation for consistently ordered matrices: given the SOR rate rho observed with
// relaxation w0, the Jacobi spectral radius mu and the optimal relaxation
double omega_from_rate(double rho, double w0)
{
    if (!(rho > 0.0) || rho >= 1.0) return w0;
    const double lam = rho;
    double mu = (lam + w0 - 1.0) / (w0 * std::sqrt(lam));
    mu = std::min(std::max(mu, 0.0), 0.9999);
    return 2.0 / (1.0 + std::sqrt(1.0 - mu * mu));
}

// The batch's stream is idle.  Up to kBatchCache bytes stay with the batch for the grids that
// join next (64 served requests at once: 302 solves/s, 285 with every block handed back); with
// more, all go where every pool can take them and sg_trim frees them.  In the batch's pool
// they would stay as long as the batch lives, which a server's does.
constexpr size_t kBatchCache = 64 << 20;

void free_fused(sg_batch *b, sg_batch::Entry &en)
{
    b->pool.free(en.x2);
    b->pool.free(en.nb);
    if (b->pool.cached_bytes() > kBatchCache) b->pool.release_cached();
    en.x2 = nullptr;
    en.nb = nullptr;
}

// What the batch keeps for a grid's fused sweeps, when the grid joins and before each step: a
// program may change a live grid between two steps, and the second buffer and the neighbour
// table are those of one chunk set.  Fused sweeps keep e = 0 where no point is, and take 2.1 KB
// a chunk of the batch's memory; a grid that does not fit makes its steps run half sweeps.
int fused_state(sg_batch *b, sg_batch::Entry &en)
{
    sg_grid *g = en.g;
    const sg_poisson_params &p = b->p;
    const bool changed = en.chunks_gen != g->chunks_gen;
    if (changed) {
        if (!g->nn_valid[SG_NN_STAR]) {
            const int rc = find_neighbours_impl(g, SG_NN_STAR);
            if (rc) return rc;
        }
        // the grid's own queued work must be done before the batch stream uses it
        SG_HIP(hipStreamSynchronize(g->stream));
    }
    static const unsigned char zero[8] = {};
    const bool fits = p.mode == SG_POISSON_MIXED && g->nchunks > 0 && g->nchunks < (1 << 21) - 1 &&
                      memcmp(g->bg[p.e_prop], zero, sizeof(float)) == 0;
    if (!changed && (fits || !en.x2)) return SG_OK;
    ++b->version;
    if (en.x2) {
        SG_HIP(hipStreamSynchronize(b->stream));  // sweeps of the last step
        free_fused(b, en);
    }
    en.prep = false;
    en.chunks_gen = g->chunks_gen;
    if (!fits) return SG_OK;
    en.x2 = (float *)b->pool.alloc((size_t)(g->nchunks + 1) * 512 * sizeof(float));
    en.nb = (int32_t *)b->pool.alloc((size_t)g->nchunks * kNb * sizeof(int32_t));
    if (!en.x2 || !en.nb) free_fused(b, en);
    en.prep = en.x2 != nullptr;
    return SG_OK;
}

// after the wait for the norms that decide it
void retire(sg_batch *b, size_t i, int converged)
{
    sg_batch::Entry &en = b->live[i];
    sg_poisson_result r;
    r.converged = converged;
    r.outer = en.outer;
    r.sweeps = en.sweeps;
    r.rel_residual = en.rel;
    r.omega = en.omega;
    r.solution_prop = en.cur_u;
    b->done.emplace_back(en.tag, r);
    free_fused(b, en);
}

}  // namespace

extern "C" {

int sg_batch_create(const sg_poisson_params *p, void *stream, sg_batch **out)
{
    if (!p || !out) return fail(SG_E_ARG, "null argument");
    if (p->mode != SG_POISSON_MIXED && p->mode != SG_POISSON_PLAIN_FP64) return fail(SG_E_ARG, "unknown mode");
    if (!(p->tol > 0.0)) return fail(SG_E_ARG, "tolerance must be positive");
    sg_batch *b = new sg_batch();
    b->p = *p;
    if (b->p.omega0 <= 0.0) b->p.omega0 = 1.5;
    if (b->p.first_sweeps <= 0) b->p.first_sweeps = 24;
    if (b->p.max_sweeps <= 0) b->p.max_sweeps = 20000;
    if (b->p.max_outer <= 0) b->p.max_outer = 100;
    if (b->p.inner_target <= 0.0) b->p.inner_target = (p->mode == SG_POISSON_MIXED) ? 1e-5 : 1e-3;
    b->stream = (hipStream_t)stream;
    if (!b->stream) {
        // stream capture is not possible on the legacy null stream; grids queued on it are
        // synchronized in sg_batch_add before the batch stream uses them
        hipError_t e = hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking);
        if (e != hipSuccess) {
            delete b;
            return fail(SG_E_HIP, std::string("hipStreamCreateWithFlags: ") + hipGetErrorString(e));
        }
        b->own_stream = true;
    }
    *out = b;
    return SG_OK;
}

int sg_batch_destroy(sg_batch *b)
{
    if (!b) return SG_OK;
    (void)hipStreamSynchronize(b->stream);
    hipStream_t own = b->own_stream ? b->stream : nullptr;
    delete b;
    if (own) (void)hipStreamDestroy(own);
    return SG_OK;
}

int sg_batch_add(sg_batch *b, sg_grid *g, int64_t tag, double tol)
{
    if (!b || !g) return fail(SG_E_ARG, "null argument");
    if (g->dim != 3 || g->edge != 8) return fail(SG_E_ARG, "batched Poisson solves need 3D grids with 8^3 chunks");
    const sg_poisson_params &p = b->p;
    const bool mixed = p.mode == SG_POISSON_MIXED;
    auto need = [&](int prop, int dt) { return prop >= 0 && prop < g->np && g->dt[prop] == dt; };
    if (!need(p.u_prop, SG_F64) || !need(p.f_prop, SG_F64) ||
        (mixed && (!need(p.u2_prop, SG_F64) || !need(p.e_prop, SG_F32) || !need(p.r_prop, SG_F32))))
        return fail(SG_E_ARG, "grid properties do not match the solver layout (u, u2, f: f64; e, r: f32)");
    sg_batch::Entry en;
    en.g = g;
    en.tag = tag;
    en.cur_u = p.u_prop;
    en.omega = (p.omega > 0.0) ? p.omega : p.omega0;
    en.inner = p.first_sweeps;
    en.tol = (tol > 0.0) ? tol : p.tol;
    en.chunks_gen = g->chunks_gen + 1;
    const int rc = fused_state(b, en);
    if (rc) return rc;
    b->live.push_back(en);
    b->dirty = true;
    ++b->version;
    return SG_OK;
}

int sg_batch_live(sg_batch *b) { return b ? (int)b->live.size() : 0; }

int sg_batch_set_tuning(sg_batch *b, int key, int64_t value)
{
    if (!b) return fail(SG_E_ARG, "null batch");
    switch (key) {
    case SG_TUNE_BATCH_WAVES:
        if (value != 0 && value != 1 && value != 2 && value != 4 && value != 8)
            return fail(SG_E_ARG, "waves must be 0 (by size), 1, 2, 4 or 8");
        b->waves = (int)value;
        break;
    case SG_TUNE_BATCH_MAX_WGS:
        if (value < 0) return fail(SG_E_ARG, "workgroup cap must be >= 0");
        b->max_wgs = value;
        break;
    default: return fail(SG_E_ARG, "unknown tuning key");
    }
    ++b->version;  // the captured sweep graph has the old launch shape
    return SG_OK;
}

// One outer iteration for every live grid: residual (+ defect correction in the mixed
// form), convergence check and retirement, then the inner sweeps of the survivors.
int sg_batch_step(sg_batch *b)
{
    if (!b) return fail(SG_E_ARG, "null batch");
    if (b->live.empty()) return SG_OK;
    const bool mixed = b->p.mode == SG_POISSON_MIXED;
    std::vector<double> norms;
    int rc;
    for (auto &en : b->live)
        if ((rc = fused_state(b, en))) return rc;
    if ((rc = defect_and_norms(b, norms, true))) return rc;
    // convergence / retirement
    std::vector<sg_batch::Entry> keep;
    for (size_t i = 0; i < b->live.size(); ++i) {
        sg_batch::Entry &en = b->live[i];
        // the mixed defect pass wrote u + e into the other u buffer
        if (mixed) en.cur_u = (en.cur_u == b->p.u_prop) ? b->p.u2_prop : b->p.u_prop;
        if (en.norm_f < 0.0) en.norm_f = std::sqrt(norms[2 * i + 1]);
        const double rn = std::sqrt(norms[2 * i]);
        en.last_rel = en.rel;
        en.rel = (en.norm_f > 0.0) ? rn / en.norm_f : 0.0;
        if (en.rel <= en.tol) {
            retire(b, i, 1);
            continue;
        }
        if (en.outer >= b->p.max_outer || en.sweeps >= b->p.max_sweeps) {
            retire(b, i, 0);
            continue;
        }
        // after each block: omega from the SOR rate observed with the block's omega.  The
        // first block starts from the rough residual f, whose fast modes decay early, so
        // its rate underestimates the asymptotic one and omega comes out low; later blocks
        // see the slow modes and refine it.  Below the optimum the dominant SOR eigenvalue
        // is real and Young's relation applies; at or above it the estimate returns the
        // block's own omega, so omega never decreases.
        if (en.outer >= 1 && b->p.omega <= 0.0 && en.last_rel > 0.0 && en.inner > 0) {
            const double rho = std::pow(std::max(en.rel / en.last_rel, 1e-300), 1.0 / en.inner);
            en.omega = std::max(en.omega, omega_from_rate(rho, en.omega));
        }
        // next block: sweeps for the wanted reduction at the asymptotic rate omega - 1 of
        // optimal SOR; never more than the remaining reduction to the tolerance asks
        if (en.outer == 0) {
            en.inner = b->p.first_sweeps;
        } else {
            const double target = std::max(b->p.inner_target, 0.5 * en.tol / en.rel);
            en.inner = sweeps_for(std::max(en.omega - 1.0, 1e-3), target, 4, 400);
        }
        keep.push_back(en);
    }
    const bool changed = keep.size() != b->live.size();
    b->live.swap(keep);
    if (changed || b->dirty) ++b->version;
    b->dirty = false;
    if (b->live.empty()) return SG_OK;
    // one launch sequence of max(inner) sweeps covers the live set; each grid stops after
    // its own count (its tiles leave the active prefix), so a grid's iterates do not
    // depend on its batch mates
    int sweeps = 0;
    for (auto &en : b->live) sweeps = std::max(sweeps, en.inner);
    // sweep work list: grids by decreasing inner count (ties in live order)
    std::vector<int> order(b->live.size());
    for (size_t i = 0; i < order.size(); ++i) order[i] = (int)i;
    std::stable_sort(order.begin(), order.end(),
                     [&](int x, int y) { return b->live[x].inner > b->live[y].inner; });
    rc = upload_worklist(b, false, order);
    if (rc) return rc;
    rc = run_sweeps(b, sweeps, mixed);
    if (rc) return rc;
    for (auto &en : b->live) {
        en.sweeps += en.inner;
        en.outer += 1;
    }
    return SG_OK;
}

int sg_batch_poll(sg_batch *b, int64_t *tags, sg_poisson_result *results, int max, int *n)
{
    if (!b || !n) return fail(SG_E_ARG, "null argument");
    int k = 0;
    while (k < max && !b->done.empty()) {
        tags[k] = b->done.front().first;
        results[k] = b->done.front().second;
        b->done.erase(b->done.begin());
        ++k;
    }
    *n = k;
    return SG_OK;
}

int sg_poisson_solve(sg_grid *const *grids, int n, const sg_poisson_params *p, sg_poisson_result *results)
{
    if (!grids || n < 0 || !p || !results) return fail(SG_E_ARG, "null argument");
    if (n == 0) return SG_OK;
    sg_batch *b = nullptr;
    int rc = sg_batch_create(p, grids[0]->stream, &b);
    if (rc) return rc;
    for (int i = 0; i < n && !rc; ++i) rc = sg_batch_add(b, grids[i], i, 0.0);
    while (!rc && !b->live.empty()) rc = sg_batch_step(b);
    if (!rc) {
        for (auto &d : b->done) results[d.first] = d.second;
    }
    sg_batch_destroy(b);
    return rc;
}

}  // extern "C"
