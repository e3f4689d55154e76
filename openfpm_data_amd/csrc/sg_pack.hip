// sg_pack.hip -- pack / unpack / remove of sparse-grid sections for gfx950.
//
// Reference: SparseGridGpu::packRequest / packCalculate / pack / packFinalize
// (src/SparseGridGpu/SparseGridGpu.hpp:3040-3340), unpack + removeAddUnpackFinalize
// (:3492-3499, :3665-3733), remove(Box) (:3528-3531) and the kernels
// calc_exist_points_with_boxes / pack_data / last_scan_point / remove_points
// (SparseGridGpu_kernels.cuh:1235-1697).
//
// Packed form of one box, sections in this order (A = sizeof(indexT), 4 or 8):
//   uint64 n_cnk | int32 box_start[dim] | int32 grid_size[dim] | indexT ids[n_cnk]
//   | uint32 scan[n_cnk + 1], padded to A | per packed property T[n_pnt], one after the
//   other, padded to A | int16 offsets[n_pnt], padded to A | uint8 masks[n_pnt], padded to A
// ids are the (sorted) chunks holding at least one existing point inside the inclusive
// box; scan[i] is the first point of chunk i and scan[n_cnk] = n_pnt.  Points of a chunk
// are written in increasing offset (the reference's order comes from an atomic counter,
// so any order is a valid instance of its format); padding bytes are zero.
//
// Kernels: a count pass (one wave per chunk, per box: existing points inside), one scan of
// the counts and the non-empty flags of all boxes, then a write pass over all boxes (one
// wave per chunk, ballot compaction keeps offsets ascending).  Unpack expands a section
// into point records (key = packed coordinate - box start + destination start) appended to
// the insert buffer; the finalize removes the queued boxes and flushes with the unpacked
// properties taking the new values.
//
// Ghost layers are small (a few thousand points of a few per cent of the chunks), so these
// calls are bound by launches, waits and the cost of passing over chunks that meet no box:
// boxes travel as kernel arguments, one launch covers all boxes, totals and flags come back
// through pinned words, and a wave leaves a chunk outside every box after some 60
// instructions (a workgroup per chunk with 64-bit divisions in every thread took 106 us for
// 22,000 chunks in each of the count and removal passes, and 16 us a box in the write pass).
// Six ghost slabs of width 3 of a 250^3 sheet packed, removed and unpacked
// (two FP32 fields, 25,000 chunks): 1.63 -> 0.47 ms, the flush that merges them included.
#include "sg_internal.hpp"

#include <algorithm>
#include <mutex>

namespace sg {
namespace {

constexpr int kWG = 256;

struct Geom {
    int dim, edge, csz;
    int sh;     // log2 of the edge, or -1
    int ids32;  // row-major chunk ids (below 2^31): 32-bit divisions
    ChunkLin L;
};

// chunk coordinates of chunk id `id` (any value: ids of packed sections are not trusted)
__device__ inline void chunk_coords_of(const Geom &G, const int64_t *bsz, int64_t id, int64_t *bc)
{
    if (G.ids32 && (uint64_t)id < ((uint64_t)1 << 31)) {
        uint32_t t = (uint32_t)id;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            if (d >= G.dim) break;
            const uint32_t b = (uint32_t)bsz[d], q = t / b;
            bc[d] = (int64_t)(t - q * b);
            t = q;
        }
        return;
    }
    ChunkLin L = G.L;
    for (int d = 0; d < 3; ++d) L.bsz[d] = bsz[d];
    chunk_coords(L, id, bc);
}

__device__ inline void chunk_origin(const Geom &G, int64_t id, int64_t *o)
{
    chunk_coords_of(G, G.L.bsz, id, o);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (d >= G.dim) break;
        o[d] *= G.edge;
    }
}

__device__ inline void local_coord(const Geom &G, int off, int64_t *l)
{
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (d >= G.dim) break;
        if (G.sh >= 0) {
            l[d] = off & (G.edge - 1);
            off >>= G.sh;
        } else {
            l[d] = off % G.edge;
            off /= G.edge;
        }
    }
}

// up to kBoxes inclusive boxes, in the kernel arguments
constexpr int kBoxes = 32;
struct Boxes {
    int n;
    int32_t lo[kBoxes * 3], hi[kBoxes * 3];  // [n][dim]
};

// property set of a grid for kernels that write or read every property
struct PropSet {
    int np;
    void *p[kMaxProps];
    int ts[kMaxProps];
    uint64_t bg[kMaxProps];
};

__device__ inline void copy_scalar(unsigned char *dst, const unsigned char *src, int ts)
{
    // byte copies: packed property arrays follow each other without alignment
    for (int b = 0; b < ts; ++b) dst[b] = src[b];
}

// little-endian values at any address (one load where it is aligned)
__device__ inline uint32_t load_u16(const unsigned char *p)
{
    if (((uintptr_t)p & 1) == 0) return *(const uint16_t *)p;
    return (uint32_t)p[0] | ((uint32_t)p[1] << 8);
}
__device__ inline uint32_t load_u32(const unsigned char *p)
{
    if (((uintptr_t)p & 3) == 0) return *(const uint32_t *)p;
    return (uint32_t)p[0] | ((uint32_t)p[1] << 8) | ((uint32_t)p[2] << 16) | ((uint32_t)p[3] << 24);
}
__device__ inline uint64_t load_u64(const unsigned char *p)
{
    return (uint64_t)load_u32(p) | ((uint64_t)load_u32(p + 4) << 32);
}

// one value of ts bytes where both addresses are multiples of ts
__device__ inline void copy_aligned(unsigned char *dst, const unsigned char *src, int ts)
{
    switch (ts) {
    case 8: *(uint64_t *)dst = *(const uint64_t *)src; break;
    case 4: *(uint32_t *)dst = *(const uint32_t *)src; break;
    case 2: *(uint16_t *)dst = *(const uint16_t *)src; break;
    default: *dst = *src; break;
    }
}

__device__ inline void clear_slot(const PropSet &P, uint8_t *mask, int64_t slot)
{
    mask[slot] = 0;
    for (int q = 0; q < P.np; ++q)
        copy_aligned((unsigned char *)P.p[q] + slot * P.ts[q], (const unsigned char *)&P.bg[q], P.ts[q]);
}

__device__ inline bool chunk_meets_box(const Geom &G, const int64_t *org, const int32_t *lo, const int32_t *hi)
{
    bool met = true;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (d >= G.dim) break;
        met = met && org[d] + G.edge - 1 >= lo[d] && org[d] <= hi[d];
    }
    return met;
}

// The kernels over chunks give lane l of a wave the slots [l V, (l + 1) V) of its chunk, V =
// ceil(csz / 64) <= 16: their mask bytes are one load (V a template parameter where csz = 64 V;
// 0 otherwise, byte loads), and lane order is slot order.
__device__ inline int lane_slots(const Geom &G, int V) { return V > 0 ? V : (G.csz + 63) / 64; }

// the masks of the lane's slots (0 past the chunk's end) and a bit per slot with EXIST
template <int V>
__device__ inline uint32_t lane_masks(const uint8_t *__restrict__ mask, int64_t c, const Geom &G, int lane,
                                      uint32_t (&m)[4])
{
    m[0] = m[1] = m[2] = m[3] = 0;
    if constexpr (V == 1) m[0] = mask[c * 64 + lane];
    else if constexpr (V == 2) m[0] = ((const uint16_t *)mask)[c * 64 + lane];
    else if constexpr (V == 4) m[0] = ((const uint32_t *)mask)[c * 64 + lane];
    else if constexpr (V == 8) {
        const uint2 q = ((const uint2 *)mask)[c * 64 + lane];
        m[0] = q.x;
        m[1] = q.y;
    } else if constexpr (V == 16) {
        const uint4 q = ((const uint4 *)mask)[c * 64 + lane];
        m[0] = q.x;
        m[1] = q.y;
        m[2] = q.z;
        m[3] = q.w;
    } else {
        const int n = lane_slots(G, 0);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int o = lane * n + v;
            if (v < n && o < G.csz) m[v >> 2] |= (uint32_t)mask[c * G.csz + o] << (8 * (v & 3));
        }
    }
    uint32_t e = 0;
#pragma unroll
    for (int v = 0; v < (V > 0 ? V : 16); ++v) e |= ((m[v >> 2] >> (8 * (v & 3))) & SG_EXIST) << v;
    return e;
}

// bit v: slot lane V + v of the chunk at org lies in the inclusive box (lo, hi)
template <int V>
__device__ inline uint32_t lane_box_bits(const Geom &G, const int64_t *org, const int32_t *lo, const int32_t *hi, int lane)
{
    // the box in chunk coordinates, cut to [0, edge)
    int a[3] = {0, 0, 0}, b[3] = {0, 0, 0};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (d >= G.dim) break;
        const int64_t l = lo[d] - org[d], h = hi[d] - org[d];
        a[d] = l < 0 ? 0 : (l > G.edge ? G.edge : (int)l);
        b[d] = h < 0 ? -1 : (h > G.edge ? G.edge : (int)h);
    }
    const int n = lane_slots(G, V);
    uint32_t in = 0;
#pragma unroll
    for (int v = 0; v < (V > 0 ? V : 16); ++v) {
        int o = lane * n + v;
        bool ok = v < n;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            if (d >= G.dim) break;
            const int q = G.sh >= 0 ? o >> G.sh : o / G.edge, x = o - q * G.edge;
            ok = ok && x >= a[d] && x <= b[d];
            o = q;
        }
        in |= (ok ? 1u : 0u) << v;
    }
    return in;
}

// bit k of the result: the chunk at org meets box k (the lanes of the wave test a box each)
__device__ inline uint32_t boxes_met(const Geom &G, const Boxes &B, const int64_t *org, int lane)
{
    bool met = false;
    if (lane < B.n) met = chunk_meets_box(G, org, B.lo + lane * G.dim, B.hi + lane * G.dim);
    return (uint32_t)__ballot(met);
}

// existing points of every chunk inside each box of B and whether there are any: box k's
// counts at cnt[k * stride + c], its flags at flag[k * stride + c], entry n of both 0
// (calc_exist_points_with_boxes, SparseGridGpu_kernels.cuh:1351-1420).  One wave per chunk
// c <= n.
template <int V>
__global__ __launch_bounds__(kWG) void pack_count_kernel(const int64_t *__restrict__ keys, int64_t n,
                                                        const uint8_t *__restrict__ mask, Geom G, Boxes B,
                                                        uint32_t *__restrict__ cnt, uint32_t *__restrict__ flag,
                                                        int64_t stride)
{
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t c = (int64_t)blockIdx.x * (kWG / 64) + w;
    if (c > n) return;
    int64_t org[3] = {0, 0, 0};
    uint32_t met = 0;
    if (c < n) {
        chunk_origin(G, keys[c], org);
        met = boxes_met(G, B, org, lane);
    }
    uint32_t mine = 0;  // lane k: the points in box k
    if (met) {
        uint32_t m[4];
        const uint32_t e = lane_masks<V>(mask, c, G, lane, m);
        for (uint32_t left = met; left; left &= left - 1) {
            const int k = __builtin_ctz(left);
            uint32_t s = (uint32_t)__popc(e & lane_box_bits<V>(G, org, B.lo + k * G.dim, B.hi + k * G.dim, lane));
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) s += (uint32_t)__shfl_xor((int)s, o, 64);
            mine = (lane == k) ? s : mine;
        }
    }
    if (lane < B.n) {
        cnt[lane * stride + c] = mine;
        flag[lane * stride + c] = mine ? 1u : 0u;
    }
}

// scan: the exclusive scan of the count rows of all boxes followed by their flag rows (per =
// boxes * stride entries each; sums wrap, differences inside a row are exact).  Box k has
// tot[2k] points in tot[2k + 1] chunks.
__global__ void pack_totals_kernel(const uint32_t *__restrict__ scan, int64_t per, int64_t stride, int nbox,
                                   uint32_t *__restrict__ tot)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nbox) return;
    const uint32_t *p = scan + (int64_t)k * stride;
    tot[2 * k] = p[stride - 1] - p[0];
    tot[2 * k + 1] = p[per + stride - 1] - p[per];
}

// the sections of the boxes of one write launch: byte offset in the buffer, chunks, points
struct PackSections {
    int64_t at[kBoxes];
    uint32_t nc[kBoxes], np[kBoxes];
};

struct PackProps {
    int n;
    int ts[kMaxProps];
    const unsigned char *src[kMaxProps];  // grid property arrays
};

// a: a power of two
__host__ __device__ inline int64_t align_up(int64_t x, int64_t a) { return (x + a - 1) & ~(a - 1); }

// addresses of one section's arrays
struct SectionPtrs {
    unsigned char *ids, *scan, *data, *offs, *masks, *end;
};

__device__ inline SectionPtrs section_ptrs(unsigned char *s0, int dim, int A, int64_t nc, int64_t np, int psz)
{
    SectionPtrs S;
    S.ids = s0 + 8 + 8 * dim;
    S.scan = S.ids + A * nc;
    S.data = S.scan + align_up((nc + 1) * 4, A);
    S.offs = S.data + align_up(np * psz, A);
    S.masks = S.offs + align_up(np * 2, A);
    S.end = S.masks + align_up(np, A);
    return S;
}

// Write the points of every box of B at their packed positions (get_exist_points_with_boxes
// + pack_data, SparseGridGpu_kernels.cuh:1437-1697).  One wave per chunk c < n; wave n + k
// writes the header, the scan's last entry and the zero padding of box k's section.  pscan /
// cscan: the boxes' rows of the scan.
template <int V>
__global__ __launch_bounds__(kWG) void pack_write_kernel(const int64_t *__restrict__ keys, int64_t n,
                                                        const uint8_t *__restrict__ mask, Geom G, Boxes B,
                                                        const uint32_t *__restrict__ pscan,
                                                        const uint32_t *__restrict__ cscan, int64_t stride, PackProps P,
                                                        int psz, int A, PackSections X, unsigned char *buf, int32_t sz0,
                                                        int32_t sz1, int32_t sz2)
{
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t c = (int64_t)blockIdx.x * (kWG / 64) + w;
    if (c >= n + B.n) return;
    if (c >= n) {
        const int k = (int)(c - n);
        unsigned char *s0 = buf + X.at[k];
        const int64_t nc = X.nc[k], np = X.np[k];
        const SectionPtrs S = section_ptrs(s0, G.dim, A, nc, np, psz);
        // sections start at multiples of 4 bytes only: byte stores
        if (lane < 8) s0[lane] = (unsigned char)((uint64_t)nc >> (8 * lane));
        const int32_t sz[3] = {sz0, sz1, sz2};
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            if (d >= G.dim || lane >= 4) continue;
            s0[8 + 4 * d + lane] = (unsigned char)((uint32_t)B.lo[k * G.dim + d] >> (8 * lane));
            s0[8 + 4 * (G.dim + d) + lane] = (unsigned char)((uint32_t)sz[d] >> (8 * lane));
        }
        unsigned char *last = S.scan + 4 * nc;
        if (lane < 4) last[lane] = (unsigned char)((uint32_t)np >> (8 * lane));
        if (last + 4 + lane < S.data) last[4 + lane] = 0;
        if (S.data + np * psz + lane < S.offs) S.data[np * psz + lane] = 0;
        if (S.offs + np * 2 + lane < S.masks) S.offs[np * 2 + lane] = 0;
        if (S.masks + np + lane < S.end) S.masks[np + lane] = 0;
        return;
    }
    // lane k: chunk c's first point and place in box k's section
    uint32_t start = 0, cnt = 0, slot = 0;
    if (lane < B.n) {
        const uint32_t *row = pscan + lane * stride;
        const uint32_t v = row[c];
        cnt = row[c + 1] - v;
        start = v - row[0];
        slot = cscan[lane * stride + c] - cscan[lane * stride];
    }
    const uint32_t any = (uint32_t)__ballot(cnt != 0);
    if (any == 0) return;
    const int64_t key = keys[c];
    int64_t org[3] = {0, 0, 0};
    chunk_origin(G, key, org);
    uint32_t m[4];
    const uint32_t e = lane_masks<V>(mask, c, G, lane, m);
    for (uint32_t left = any; left; left &= left - 1) {
        const int k = __builtin_ctz(left);
        const uint32_t st = (uint32_t)__shfl((int)start, k, 64), sl = (uint32_t)__shfl((int)slot, k, 64);
        const int64_t np = X.np[k];
        const SectionPtrs S = section_ptrs(buf + X.at[k], G.dim, A, X.nc[k], np, psz);
        if (lane < A) S.ids[(int64_t)sl * A + lane] = (unsigned char)((uint64_t)key >> (8 * lane));
        if (lane < 4) S.scan[(int64_t)sl * 4 + lane] = (unsigned char)(st >> (8 * lane));
        const uint32_t in = e & lane_box_bits<V>(G, org, B.lo + k * G.dim, B.hi + k * G.dim, lane);
        // the lanes' first points: exclusive prefix of their counts
        const uint32_t own = (uint32_t)__popc(in);
        uint32_t inc = own;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t u = (uint32_t)__shfl_up((int)inc, o, 64);
            if (lane >= o) inc += u;
        }
        int64_t j = (int64_t)st + inc - own;
        const int o0 = lane * lane_slots(G, V);
        for (uint32_t b = in; b; b &= b - 1, ++j) {
            const int v = __builtin_ctz(b), o = o0 + v;
            const int64_t slot_pt = c * G.csz + o;
            unsigned char *d = S.data;
            for (int q = 0; q < P.n; ++q) {
                const int ts = P.ts[q];
                // arrays follow each other without alignment
                if (((uintptr_t)d & (uintptr_t)(ts - 1)) == 0) copy_aligned(d + j * ts, P.src[q] + slot_pt * ts, ts);
                else copy_scalar(d + j * ts, P.src[q] + slot_pt * ts, ts);
                d += np * ts;
            }
            const int16_t o16 = (int16_t)o;
            if (((uintptr_t)S.offs & 1) == 0) ((int16_t *)S.offs)[j] = o16;
            else copy_scalar(S.offs + 2 * j, (const unsigned char *)&o16, 2);
            const uint32_t mw = v < 8 ? (v < 4 ? m[0] : m[1]) : (v < 12 ? m[2] : m[3]);
            S.masks[j] = (uint8_t)(mw >> (8 * (v & 3)));
        }
    }
}

struct UnpackIn {
    const unsigned char *buf;
    int64_t avail;
    int A, psz;                 // bytes of a chunk id, of a point's packed values
    int off[kMaxProps];         // per grid property: packed bytes per point before its array, -1: not packed
    int32_t dst_lo[3];
};

// words of a section's report (pinned host memory)
enum { kUpChunks = 0, kUpStart = 2, kUpSize = 5, kUpPoints = 8, kUpState = 9, kUpBad = 10 };

// One packed section in device memory: packed chunk i -> point records at scan[i] .. of the
// record arrays (copy_packed_data_to_chunks, SparseGridGpu_kernels.cuh:1591-1632; mask |=
// EXIST), one wave per chunk (grid stride).  Every wave reads the header itself, so the host
// needs no look at the section before the launch: it learns n_cnk, box start, grid size,
// n_pnt, the state (bit 0: the chunk list and scan lie inside the section; bit 1: the
// records were written, as they are when the section is whole and `room` takes its points)
// and whether a record was bad from the report, in one wait.
__global__ __launch_bounds__(kWG) void unpack_section_kernel(UnpackIn U, Geom G, int64_t sz0, int64_t sz1, int64_t sz2,
                                                            PropSet P, int64_t *__restrict__ rkey,
                                                            uint8_t *__restrict__ rmask, int64_t room,
                                                            uint32_t *__restrict__ rep)
{
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t first = (int64_t)blockIdx.x * (kWG / 64) + w, hsz = 8 + 8 * G.dim;
    // a section may start at any address
    const uint64_t nc = load_u64(U.buf);
    int32_t bstart[3] = {0, 0, 0}, psize[3] = {1, 1, 1};
    bool sizes = true;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (d >= G.dim) break;
        bstart[d] = (int32_t)load_u32(U.buf + 8 + 4 * d);
        psize[d] = (int32_t)load_u32(U.buf + 8 + 4 * (G.dim + d));
        sizes = sizes && psize[d] > 0;
    }
    // the chunk list and the scan lie inside (nc < avail first: no overflow below)
    const bool whole = nc < (uint64_t)U.avail && U.avail >= hsz + U.A * (int64_t)nc + ((int64_t)nc + 1) * 4;
    const int64_t n_cnk = (int64_t)nc;
    const uint32_t np = whole ? load_u32(U.buf + hsz + U.A * n_cnk + n_cnk * 4) : 0u;
    const int64_t n_pnt = np;
    const unsigned char *ids = U.buf + hsz, *scan = ids + U.A * n_cnk;
    const unsigned char *data = scan + align_up((n_cnk + 1) * 4, U.A);
    const unsigned char *offs = data + align_up(n_pnt * U.psz, U.A);
    const unsigned char *end = offs + align_up(n_pnt * 2, U.A) + align_up(n_pnt, U.A);
    const bool go = whole && sizes && end - U.buf <= U.avail && n_pnt <= room;
    if (first == 0 && lane == 0) {
        rep[kUpChunks] = (uint32_t)nc;
        rep[kUpChunks + 1] = (uint32_t)(nc >> 32);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            if (d >= G.dim) break;
            rep[kUpStart + d] = (uint32_t)bstart[d];
            rep[kUpSize + d] = (uint32_t)psize[d];
        }
        rep[kUpPoints] = np;
        rep[kUpState] = (whole ? 1u : 0u) | (go ? 2u : 0u);
    }
    if (!go) return;
    int64_t pbsz[3] = {1, 1, 1};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (d >= G.dim) break;
        pbsz[d] = ((int64_t)psize[d] + G.edge - 1) / G.edge;
    }
    const int64_t sz[3] = {sz0, sz1, sz2}, stride = (int64_t)gridDim.x * (kWG / 64);
    for (int64_t i = first; i < n_cnk; i += stride) {
        const int64_t id = U.A == 8 ? (int64_t)load_u64(ids + i * 8) : (int64_t)(int32_t)load_u32(ids + i * 4);
        const int64_t j0 = load_u32(scan + 4 * i), j1 = load_u32(scan + 4 * i + 4);
        // chunk coordinates in the packing grid (same linearizer, its own chunk counts)
        int64_t bc[3] = {0, 0, 0};
        chunk_coords_of(G, pbsz, id, bc);
        // a malformed section (scan not starting at 0, not increasing or past n_pnt) is
        // refused, not followed: the records [0, n_pnt) are then exactly the chunks' ranges
        if (j0 > j1 || j1 > n_pnt || (i == 0 && j0 != 0)) {
            if (lane == 0) rep[kUpBad] = 1;
            return;
        }
        for (int64_t j = j0 + lane; j < j1; j += 64) {
            const int off = (int)load_u16(offs + 2 * j);
            int64_t l[3] = {0, 0, 0}, c[3] = {0, 0, 0};
            local_coord(G, off, l);
            bool ok = off < G.csz;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                if (d >= G.dim) break;
                c[d] = bc[d] * G.edge + l[d] + ((int64_t)U.dst_lo[d] - bstart[d]);
                ok = ok && c[d] >= 0 && c[d] < sz[d];
            }
            if (!ok) {
                rep[kUpBad] = 1;
                rkey[j] = 0;
                rmask[j] = 0;
                continue;
            }
            int64_t cb[3] = {0, 0, 0}, lo = 0;
#pragma unroll
            for (int d = 2; d >= 0; --d) {
                if (d >= G.dim) continue;
                cb[d] = G.sh >= 0 ? c[d] >> G.sh : c[d] / G.edge;
                lo = lo * G.edge + (c[d] - cb[d] * G.edge);
            }
            rkey[j] = chunk_id(G.L, cb) * G.csz + lo;
            rmask[j] = SG_EXIST;
            for (int q = 0; q < P.np; ++q) {
                const int ts = P.ts[q];
                unsigned char *dst = (unsigned char *)P.p[q] + j * ts;
                const unsigned char *src = data + n_pnt * U.off[q];
                if (U.off[q] < 0) copy_aligned(dst, (const unsigned char *)&P.bg[q], ts);
                else if (((uintptr_t)src & (uintptr_t)(ts - 1)) == 0) copy_aligned(dst, src + j * ts, ts);
                else copy_scalar(dst, src + j * ts, ts);
            }
        }
    }
}

// remove_points (SparseGridGpu_kernels.cuh:1301-1346): existing points inside a queued box
// get mask 0 (and the background value)
// one wave per chunk
template <int V>
__global__ __launch_bounds__(kWG) void remove_boxes_kernel(const int64_t *__restrict__ keys, int64_t n,
                                                          uint8_t *mask, Geom G, Boxes B, PropSet P)
{
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t c = (int64_t)blockIdx.x * (kWG / 64) + w;
    if (c >= n) return;
    int64_t org[3] = {0, 0, 0};
    chunk_origin(G, keys[c], org);
    const uint32_t met = boxes_met(G, B, org, lane);
    if (met == 0) return;
    uint32_t m[4];
    const uint32_t e = lane_masks<V>(mask, c, G, lane, m);
    uint32_t in = 0;
    for (uint32_t left = met; left; left &= left - 1) {
        const int k = __builtin_ctz(left);
        in |= lane_box_bits<V>(G, org, B.lo + k * G.dim, B.hi + k * G.dim, lane);
    }
    const int64_t s0 = c * G.csz + lane * lane_slots(G, V);
    for (uint32_t b = e & in; b; b &= b - 1) clear_slot(P, mask, s0 + __builtin_ctz(b));
}

__device__ inline int64_t lower_bound_keys(const int64_t *a, int64_t n, int64_t x)
{
    int64_t lo = 0, hi = n;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (a[mid] < x) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// device remove(coord) (BlockMapGpu_ker.cuh:322-332) for a list of point keys
__global__ void remove_points_kernel(const int64_t *__restrict__ keys, int64_t n, uint8_t *__restrict__ mask,
                                     const int64_t *__restrict__ pk, int64_t m, int csz, PropSet P)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    const int64_t k = pk[i];
    if (k < 0) return;
    const int64_t c = lower_bound_keys(keys, n, k / csz);
    if (c < n && keys[c] == k / csz) clear_slot(P, mask, c * csz + k % csz);
}

Geom geom_of(const sg_grid *g)
{
    Geom G;
    G.dim = g->dim;
    G.edge = g->edge;
    G.csz = g->csz;
    G.sh = -1;
    for (int b = 1; b < 11; ++b)
        if ((1 << b) == g->edge) G.sh = b;
    G.L = chunk_lin(g);
    // chunk counts below 2^31 (sg_create) give row-major ids below 2^31
    G.ids32 = !G.L.zorder;
    return G;
}

PropSet grid_props(sg_grid *g)
{
    PropSet P;
    P.np = g->np;
    for (int q = 0; q < g->np; ++q) {
        P.p[q] = g->d_prop[q];
        P.ts[q] = g->ts[q];
        P.bg[q] = 0;
        memcpy(&P.bg[q], g->bg[q], g->ts[q]);
    }
    return P;
}

int check_pack_args(const sg_grid *g, int nbox, const int32_t *lo, const int32_t *hi, int nprop,
                    const int32_t *props, int A)
{
    if (nbox < 0 || nprop < 0) return fail(SG_E_ARG, "negative count");
    if (nbox > 0 && (!lo || !hi)) return fail(SG_E_ARG, "null boxes");
    if (nprop > 0 && !props) return fail(SG_E_ARG, "null property list");
    if (nprop > kMaxProps) return fail(SG_E_ARG, "more properties than a grid can have");
    if (A != 4 && A != 8) return fail(SG_E_ARG, "index_bytes must be 4 or 8");
    for (int q = 0; q < nprop; ++q)
        if (props[q] < 0 || props[q] >= g->np) return fail(SG_E_ARG, "bad property");
    if (g->csz > 32768) return fail(SG_E_ARG, "chunk too large for 16-bit offsets");
    return SG_OK;
}

int64_t point_bytes(const sg_grid *g, int nprop, const int32_t *props)
{
    int64_t s = 0;
    for (int q = 0; q < nprop; ++q) s += g->ts[props[q]];
    return s;
}

int64_t section_bytes(const sg_grid *g, int64_t n_cnk, int64_t n_pnt, int64_t psz, int A)
{
    return 8 + 2 * g->dim * 4 + A * n_cnk + align_up((n_cnk + 1) * 4, A) + align_up(n_pnt * psz, A) +
           align_up(n_pnt * 2, A) + align_up(n_pnt, A);
}

// boxes [k0, k0 + kBoxes) of a list as kernel arguments
Boxes box_args(int dim, int nbox, const int32_t *lo, const int32_t *hi, int k0)
{
    Boxes B;
    B.n = std::min(kBoxes, nbox - k0);
    memcpy(B.lo, lo + (size_t)k0 * dim, (size_t)B.n * dim * 4);
    memcpy(B.hi, hi + (size_t)k0 * dim, (size_t)B.n * dim * 4);
    return B;
}

// f(std::integral_constant<int, V>) for the lane runs of the grid's chunks
template <typename F> void with_lane_run(const sg_grid *g, F &&f)
{
    switch (g->csz) {
    case 64: f(std::integral_constant<int, 1>()); break;
    case 128: f(std::integral_constant<int, 2>()); break;
    case 256: f(std::integral_constant<int, 4>()); break;
    case 512: f(std::integral_constant<int, 8>()); break;
    case 1024: f(std::integral_constant<int, 16>()); break;
    default: f(std::integral_constant<int, 0>()); break;
    }
}

unsigned chunk_waves(int64_t n) { return (unsigned)((n + kWG / 64 - 1) / (kWG / 64)); }

// Per box (rows of stride = chunks + 1 entries) the scan of the point counts, then (from
// entry per = nbox * stride) of the non-empty flags, in one exclusive scan over all rows
// (in place), and the boxes' totals.
struct PackPlan {
    int64_t stride = 0, per = 0;
    uint32_t *scan = nullptr;
    std::vector<int64_t> n_cnk, n_pnt;
};

// the counts of every box in pl.scan and, after the caller's scan of them, their totals in
// d_tot [2 * nbox] (queued on the grid's stream)
int pack_counts(sg_grid *g, int nbox, const int32_t *lo, const int32_t *hi, int64_t stride, uint32_t *rows)
{
    const int64_t n = g->nchunks, per = nbox * stride;
    for (int k0 = 0; k0 < nbox; k0 += kBoxes) {
        with_lane_run(g, [&](auto v) {
            hipLaunchKernelGGL(pack_count_kernel<decltype(v)::value>, dim3(chunk_waves(n + 1)), dim3(kWG), 0, g->stream,
                               g->d_keys, n, g->d_mask, geom_of(g), box_args(g->dim, nbox, lo, hi, k0),
                               rows + k0 * stride, rows + per + k0 * stride, stride);
        });
        SG_HIP(hipGetLastError());
    }
    return SG_OK;
}

int plan_pack(sg_grid *g, int nbox, const int32_t *lo, const int32_t *hi, PackPlan &pl)
{
    const int64_t n = g->nchunks;
    pl.stride = n + 1;
    pl.per = nbox * pl.stride;
    pl.n_cnk.assign(nbox, 0);
    pl.n_pnt.assign(nbox, 0);
    if (nbox == 0) return SG_OK;
    int rc;
    DevBuf &b_cnt = g->scratch[1];
    if ((rc = ensure(g->pool, b_cnt, (size_t)pl.per * 2 * sizeof(uint32_t) + (size_t)nbox * 2 * sizeof(uint32_t) + 64)))
        return rc;
    pl.scan = (uint32_t *)b_cnt.p;
    if ((rc = pack_counts(g, nbox, lo, hi, pl.stride, pl.scan))) return rc;
    if ((rc = exclusive_scan_u32(g, pl.scan, pl.scan, 2 * pl.per, nullptr))) return rc;
    // totals: straight to the pinned words when they fit
    uint32_t *hw = host_words(g);
    if (!hw) return fail(SG_E_OOM, "pinned host allocation failed");
    const bool pinned = nbox <= 8;
    uint32_t *tot = pinned ? hw : pl.scan + 2 * pl.per;
    hipLaunchKernelGGL(pack_totals_kernel, dim3(grid_1d(nbox, 64)), dim3(64), 0, g->stream, pl.scan, pl.per, pl.stride,
                       nbox, tot);
    SG_HIP(hipGetLastError());
    std::vector<uint32_t> h(pinned ? 0 : 2 * (size_t)nbox);
    if (!pinned)
        SG_HIP(hipMemcpyAsync(h.data(), tot, (size_t)nbox * 2 * sizeof(uint32_t), hipMemcpyDeviceToHost, g->stream));
    SG_HIP(hipStreamSynchronize(g->stream));
    const uint32_t *t = pinned ? hw : h.data();
    for (int k = 0; k < nbox; ++k) {
        pl.n_pnt[k] = t[2 * k];
        pl.n_cnk[k] = t[2 * k + 1];
    }
    return SG_OK;
}

// write the packed sections of the boxes to the device buffer buf (cap bytes) from the
// scanned rows of a plan; queued on the grid's stream, allocates nothing
int pack_sections(sg_grid *g, int nbox, const int32_t *lo, const int32_t *hi, int nprop, const int32_t *props, int A,
                  unsigned char *buf, int64_t cap, int64_t stride, const uint32_t *scan, const int64_t *n_cnk,
                  const int64_t *n_pnt)
{
    const int64_t psz = point_bytes(g, nprop, props), n = g->nchunks, per = nbox * stride;
    PackProps P;
    P.n = nprop;
    for (int q = 0; q < nprop; ++q) {
        P.ts[q] = g->ts[props[q]];
        P.src[q] = (const unsigned char *)g->d_prop[props[q]];
    }
    int64_t at = 0;
    for (int k0 = 0; k0 < nbox; k0 += kBoxes) {
        const Boxes B = box_args(g->dim, nbox, lo, hi, k0);
        PackSections X;
        for (int k = 0; k < B.n; ++k) {
            X.at[k] = at;
            X.nc[k] = (uint32_t)n_cnk[k0 + k];
            X.np[k] = (uint32_t)n_pnt[k0 + k];
            at += section_bytes(g, n_cnk[k0 + k], n_pnt[k0 + k], psz, A);
            if (at > cap) return fail(SG_E_RANGE, "pack buffer too small");
        }
        with_lane_run(g, [&](auto v) {
            hipLaunchKernelGGL(pack_write_kernel<decltype(v)::value>, dim3(chunk_waves(n + B.n)), dim3(kWG), 0, g->stream,
                               g->d_keys, n, g->d_mask, geom_of(g), B, scan + k0 * stride, scan + per + k0 * stride,
                               stride, P, (int)psz, A, X, buf, (int32_t)g->sz[0], (int32_t)g->sz[1], (int32_t)g->sz[2]);
        });
        SG_HIP(hipGetLastError());
    }
    return SG_OK;
}

// the packed sections from a plan, complete when the call returns
int pack_into_device(sg_grid *g, int nbox, const int32_t *lo, const int32_t *hi, int nprop, const int32_t *props, int A,
                     unsigned char *buf, int64_t cap, const PackPlan &pl)
{
    int rc = pack_sections(g, nbox, lo, hi, nprop, props, A, buf, cap, pl.stride, pl.scan, pl.n_cnk.data(),
                           pl.n_pnt.data());
    if (rc) return rc;
    SG_HIP(hipStreamSynchronize(g->stream));
    return SG_OK;
}

// ---- pack without device allocation (sg_pack_noalloc) -----------------------------
// The count / scan temporaries live in one static device array per GPU.  Host code never
// uses the array's name as an address: its device address comes from hipGetSymbolAddress,
// taken once per device with that device current, and only that address is passed on.
static __device__ __align__(256) unsigned char scratch[SG_PACK_NOALLOC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {};

// device address of `scratch` on the current device
int noalloc_scratch(void **out)
{
    int dev = -1;
    SG_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(SG_E_ARG, "device index beyond the scratch table");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(SG_E_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return SG_OK;
}

constexpr size_t round256(size_t b) { return (b + 255) & ~(size_t)255; }

// scratch bytes a pack of nbox boxes over n chunks may use (the call's documented limit:
// box corners, four rows of every box, per-box totals and a scan workspace); two rows of
// every box, the totals and the workspace of one scan over the rows are in use
size_t noalloc_pack_bytes(int nbox, int dim, int64_t n)
{
    const size_t stride = (size_t)n + 1;
    return round256((size_t)2 * nbox * dim * 4) + round256((size_t)4 * nbox * stride * 4) +
           round256((size_t)2 * nbox * 4) + round256(scan_ws_words((int64_t)stride) * 4);
}

}  // namespace
}  // namespace sg

using namespace sg;

extern "C" {

int sg_pack_size(sg_grid *g, int nbox, const int32_t *lo, const int32_t *hi, int nprop, const int32_t *props,
                 int index_bytes, int64_t *bytes)
{
    if (!g || !bytes) return fail(SG_E_ARG, "null argument");
    int rc = check_pack_args(g, nbox, lo, hi, nprop, props, index_bytes);
    if (rc) return rc;
    PackPlan pl;
    if ((rc = plan_pack(g, nbox, lo, hi, pl))) return rc;
    const int64_t psz = point_bytes(g, nprop, props);
    int64_t tot = 0;
    for (int k = 0; k < nbox; ++k) tot += section_bytes(g, pl.n_cnk[k], pl.n_pnt[k], psz, index_bytes);
    *bytes = tot;
    return SG_OK;
}

int sg_pack(sg_grid *g, int nbox, const int32_t *lo, const int32_t *hi, int nprop, const int32_t *props,
            int index_bytes, void *buf, int64_t cap, int mem)
{
    if (!g || (!buf && cap > 0)) return fail(SG_E_ARG, "null argument");
    int rc = check_pack_args(g, nbox, lo, hi, nprop, props, index_bytes);
    if (rc) return rc;
    PackPlan pl;
    if ((rc = plan_pack(g, nbox, lo, hi, pl))) return rc;
    const int64_t psz = point_bytes(g, nprop, props);
    int64_t tot = 0;
    for (int k = 0; k < nbox; ++k) tot += section_bytes(g, pl.n_cnk[k], pl.n_pnt[k], psz, index_bytes);
    if (tot > cap) return fail(SG_E_RANGE, "pack buffer too small");
    if (mem == SG_MEM_DEVICE) {
        rc = pack_into_device(g, nbox, lo, hi, nprop, props, index_bytes, (unsigned char *)buf, cap, pl);
        return rc;
    }
    DevBuf &st = g->scratch[2];
    if ((rc = ensure(g->pool, st, (size_t)tot + 64))) return rc;
    if ((rc = pack_into_device(g, nbox, lo, hi, nprop, props, index_bytes, (unsigned char *)st.p, tot, pl)))
        return rc;
    SG_HIP(hipMemcpyAsync(buf, st.p, (size_t)tot, hipMemcpyDeviceToHost, g->stream));
    SG_HIP(hipStreamSynchronize(g->stream));
    return SG_OK;
}

int sg_pack_noalloc(sg_grid *g, int nbox, const int32_t *lo, const int32_t *hi, int nprop, const int32_t *props,
                    int index_bytes, void *dev_buf, int64_t cap, int64_t *written)
{
    if (!g || !written || (!dev_buf && cap > 0)) return fail(SG_E_ARG, "null argument");
    int rc = check_pack_args(g, nbox, lo, hi, nprop, props, index_bytes);
    if (rc) return rc;
    if (nbox > SG_PACK_NOALLOC_MAX_BOXES)
        return fail(SG_E_RANGE, "sg_pack_noalloc: " + std::to_string(nbox) + " boxes, at most " +
                                    std::to_string(SG_PACK_NOALLOC_MAX_BOXES));
    const int64_t n = g->nchunks, stride = n + 1;
    const size_t need = noalloc_pack_bytes(nbox, g->dim, n);
    if (need > (size_t)SG_PACK_NOALLOC_SCRATCH_BYTES)
        return fail(SG_E_RANGE, "sg_pack_noalloc: " + std::to_string(nbox) + " boxes over " + std::to_string(n) +
                                    " chunks need " + std::to_string(need) + " scratch bytes, more than the " +
                                    std::to_string((size_t)SG_PACK_NOALLOC_SCRATCH_BYTES) + " reserved");
    *written = 0;
    if (nbox == 0) return SG_OK;
    void *base = nullptr;
    if ((rc = noalloc_scratch(&base))) return rc;
    // carve the scratch: count and flag rows (scanned in place) | totals | scan workspace
    const int64_t per = nbox * stride;
    const size_t rows_bytes = round256((size_t)per * 2 * 4), tot_bytes = round256((size_t)2 * nbox * 4);
    const size_t ws_words = scan_ws_words(2 * per);
    if (rows_bytes + tot_bytes + ws_words * 4 > (size_t)SG_PACK_NOALLOC_SCRATCH_BYTES)
        return fail(SG_E_RANGE, "sg_pack_noalloc: scratch too small");
    uint32_t *scan = (uint32_t *)base;
    uint32_t *d_tot = (uint32_t *)((unsigned char *)base + rows_bytes);
    uint32_t *ws = (uint32_t *)((unsigned char *)base + rows_bytes + tot_bytes);
    if ((rc = pack_counts(g, nbox, lo, hi, stride, scan))) return rc;
    if ((rc = exclusive_scan_u32_ws(g->stream, scan, scan, 2 * per, nullptr, ws, ws_words))) return rc;
    hipLaunchKernelGGL(pack_totals_kernel, dim3(grid_1d(nbox, 64)), dim3(64), 0, g->stream, scan, per, stride, nbox,
                       d_tot);
    SG_HIP(hipGetLastError());
    uint32_t h_tot[2 * SG_PACK_NOALLOC_MAX_BOXES];
    SG_HIP(hipMemcpyAsync(h_tot, d_tot, (size_t)2 * nbox * 4, hipMemcpyDeviceToHost, g->stream));
    SG_HIP(hipStreamSynchronize(g->stream));
    int64_t n_pnt[SG_PACK_NOALLOC_MAX_BOXES], n_cnk[SG_PACK_NOALLOC_MAX_BOXES];
    const int64_t psz = point_bytes(g, nprop, props);
    int64_t tot = 0;
    for (int k = 0; k < nbox; ++k) {
        n_pnt[k] = h_tot[2 * k];
        n_cnk[k] = h_tot[2 * k + 1];
        tot += section_bytes(g, n_cnk[k], n_pnt[k], psz, index_bytes);
    }
    if (tot > cap) return fail(SG_E_RANGE, "pack buffer too small: " + std::to_string(tot) + " bytes needed");
    if ((rc = pack_sections(g, nbox, lo, hi, nprop, props, index_bytes, (unsigned char *)dev_buf, cap, stride, scan,
                            n_cnk, n_pnt)))
        return rc;
    SG_HIP(hipStreamSynchronize(g->stream));
    *written = tot;
    return SG_OK;
}

int sg_unpack(sg_grid *g, const void *buf, int64_t avail, int mem, const int32_t *dst_lo, int nprop,
              const int32_t *props, int index_bytes, int64_t *consumed)
{
    if (!g || !buf || !dst_lo || !consumed) return fail(SG_E_ARG, "null argument");
    int rc = check_pack_args(g, 0, nullptr, nullptr, nprop, props, index_bytes);
    if (rc) return rc;
    const int A = index_bytes;
    const int64_t hsz = 8 + 2 * g->dim * 4;
    if (avail < hsz) return fail(SG_E_RANGE, "packed section truncated");
    uint32_t *hw = host_words(g);
    if (!hw) return fail(SG_E_OOM, "pinned host allocation failed");
    const int64_t psz = point_bytes(g, nprop, props);
    UnpackIn U;
    U.A = A;
    U.psz = (int)psz;
    for (int p = 0; p < kMaxProps; ++p) U.off[p] = -1;
    for (int pi = 0, o = 0; pi < nprop; ++pi) {
        U.off[props[pi]] = o;
        o += g->ts[props[pi]];
    }
    for (int d = 0; d < 3; ++d) U.dst_lo[d] = d < g->dim ? dst_lo[d] : 0;
    // records go to the insert buffer at `at` (room for `room` of them); values of the
    // properties not unpacked are the background (the finalize keeps the old values there)
    int64_t at = g->ins_n, room = g->ins_cap - g->ins_n;
    if (g->cins_n > 0 || g->pins_n > 0) room = 0;  // converted to point records first, below
    auto launch = [&](const unsigned char *s0, int64_t bytes) -> int {
        PropSet R;
        R.np = g->np;
        for (int p = 0; p < g->np; ++p) {
            R.p[p] = (unsigned char *)g->d_ins_val[p] + at * g->ts[p];
            R.ts[p] = g->ts[p];
            R.bg[p] = 0;
            memcpy(&R.bg[p], g->bg[p], g->ts[p]);
        }
        U.buf = s0;
        U.avail = bytes;
        // the report: the flag is written only by a thread that meets a bad record
        hw[kUpState] = hw[kUpBad] = 0;
        const unsigned grid = std::min<unsigned>(1024, chunk_waves(std::max<int64_t>(1, bytes / (A + 4))));
        hipLaunchKernelGGL(unpack_section_kernel, dim3(grid), dim3(kWG), 0, g->stream, U, geom_of(g), g->sz[0], g->sz[1],
                           g->sz[2], R, g->d_ins_key + at, g->d_ins_mask + at, room, hw);
        SG_HIP(hipGetLastError());
        SG_HIP(hipStreamSynchronize(g->stream));
        return SG_OK;
    };
    const unsigned char *s0 = (const unsigned char *)buf;
    int64_t nc = 0, sec = avail;
    uint32_t np32 = 0;
    bool whole = false, sizes = true, done = false;
    if (mem == SG_MEM_DEVICE) {
        if ((rc = launch(s0, avail))) return rc;
        nc = (int64_t)((uint64_t)hw[kUpChunks] | ((uint64_t)hw[kUpChunks + 1] << 32));
        for (int d = 0; d < g->dim; ++d) sizes = sizes && (int32_t)hw[kUpSize + d] > 0;
        np32 = hw[kUpPoints];
        whole = (hw[kUpState] & 1) != 0;
        done = (hw[kUpState] & 2) != 0;
    } else {
        memcpy(&nc, s0, 8);
        for (int d = 0; d < g->dim; ++d) {
            int32_t v;
            memcpy(&v, s0 + 8 + 4 * (g->dim + d), 4);
            sizes = sizes && v > 0;
        }
        whole = nc >= 0 && nc < avail && avail >= hsz + A * nc + (nc + 1) * 4;
        if (whole) memcpy(&np32, s0 + hsz + A * nc + nc * 4, 4);
    }
    if (!sizes) return fail(SG_E_RANGE, "bad packed grid size");
    if (!whole) return fail(SG_E_RANGE, "packed section truncated");
    const int64_t np = np32;
    const int64_t sb = section_bytes(g, nc, np, psz, A);
    if (avail < sb) return fail(SG_E_RANGE, "packed section truncated");
    if (nc == 0 && np != 0) return fail(SG_E_RANGE, "malformed packed section: points without chunks");
    *consumed = sb;
    if (np == 0) return SG_OK;
    if (!done) {
        if (mem != SG_MEM_DEVICE) {
            DevBuf &st = g->scratch[2];
            if ((rc = ensure(g->pool, st, (size_t)sb + 64))) return rc;
            SG_HIP(hipMemcpyAsync(st.p, buf, (size_t)sb, hipMemcpyHostToDevice, g->stream));
            s0 = (const unsigned char *)st.p;
            sec = sb;
        }
        if ((rc = reserve_point_records(g, np, &at))) return rc;
        room = np;
        if ((rc = launch(s0, sec))) return rc;
    }
    if (hw[kUpBad]) return fail(SG_E_RANGE, "unpacked point outside the grid or malformed packed section");
    g->ins_n = at + np;
    return SG_OK;
}

int sg_remove_box(sg_grid *g, const int32_t *lo, const int32_t *hi)
{
    if (!g || !lo || !hi) return fail(SG_E_ARG, "null argument");
    for (int d = 0; d < g->dim; ++d) {
        g->rem_lo.push_back(lo[d]);
        g->rem_hi.push_back(hi[d]);
    }
    return SG_OK;
}

int sg_remove_points(sg_grid *g, int64_t n, const int64_t *keys, int mem)
{
    if (!g || (n > 0 && !keys)) return fail(SG_E_ARG, "null argument");
    if (n <= 0 || g->nchunks == 0) return SG_OK;
    const int64_t *dk = keys;
    if (mem != SG_MEM_DEVICE) {
        int rc = ensure(g->pool, g->scratch[9], (size_t)n * 8 + 64);
        if (rc) return rc;
        SG_HIP(hipMemcpyAsync(g->scratch[9].p, keys, (size_t)n * 8, hipMemcpyHostToDevice, g->stream));
        dk = (const int64_t *)g->scratch[9].p;
    }
    g->occ_tab_valid = false;
    g->ebits_valid = false;
    hipLaunchKernelGGL(remove_points_kernel, dim3(grid_1d(n, kWG)), dim3(kWG), 0, g->stream, g->d_keys, g->nchunks,
                       g->d_mask, dk, n, g->csz, grid_props(g));
    SG_HIP(hipGetLastError());
    g->ep_valid = false;
    if (mem != SG_MEM_DEVICE) SG_HIP(hipStreamSynchronize(g->stream));  // the host keys are the caller's
    return SG_OK;
}

}  // extern "C"

namespace {

// clear the points of the boxes queued by sg_remove_box (mask 0, value background)
int remove_queued_boxes(sg_grid *g)
{
    const int nb = (int)(g->rem_lo.size() / std::max(1, g->dim));
    if (nb > 0 && g->nchunks > 0) {
        g->occ_tab_valid = false;
        g->ebits_valid = false;
        for (int k0 = 0; k0 < nb; k0 += kBoxes) {
            with_lane_run(g, [&](auto v) {
                hipLaunchKernelGGL(remove_boxes_kernel<decltype(v)::value>, dim3(chunk_waves(g->nchunks)), dim3(kWG), 0,
                                   g->stream, g->d_keys, g->nchunks, g->d_mask, geom_of(g),
                                   box_args(g->dim, nb, g->rem_lo.data(), g->rem_hi.data(), k0), grid_props(g));
            });
            SG_HIP(hipGetLastError());
        }
        g->ep_valid = false;
    }
    g->rem_lo.clear();
    g->rem_hi.clear();
    return SG_OK;
}

int check_props(sg_grid *g, int nprop, const int32_t *props)
{
    if (nprop > 0 && !props) return fail(SG_E_ARG, "null argument");
    for (int q = 0; q < nprop; ++q)
        if (props[q] < 0 || props[q] >= g->np) return fail(SG_E_ARG, "bad property");
    return SG_OK;
}

// unpacked properties: the unpacked value (left operand) wins over the old one; the
// others keep the old value (right operand), new points get the background
int flush_unpacked(sg_grid *g, int nprop, const int32_t *props)
{
    std::vector<int32_t> ops(g->np, SG_OP_RIGHT);
    for (int q = 0; q < nprop; ++q) ops[props[q]] = SG_OP_LEFT;
    return flush_impl(g, ops.data());
}

// phase 2 of removeCopyToFinalize: pack every queued section of g into one device buffer,
// then unpack each into its destination's insert buffer
int copy_sections_out(sg_grid *g, int nprop, const int32_t *props)
{
    if (g->copies.empty()) return SG_OK;
    const int n = (int)g->copies.size(), D = g->dim;
    for (const auto &c : g->copies) {
        sg_grid *d = c.dst;
        if (d->dim != D) return fail(SG_E_ARG, "copy_to: grids of different dimension");
        for (int q = 0; q < nprop; ++q)
            if (props[q] >= d->np || d->dt[props[q]] != g->dt[props[q]])
                return fail(SG_E_ARG, "copy_to: property types differ between the grids");
    }
    std::vector<int32_t> lo((size_t)n * D), hi((size_t)n * D);
    for (int k = 0; k < n; ++k)
        for (int a = 0; a < D; ++a) {
            lo[(size_t)k * D + a] = g->copies[k].lo[a];
            hi[(size_t)k * D + a] = g->copies[k].hi[a];
        }
    std::vector<int64_t> bytes(n);
    int64_t tot = 0;
    for (int k = 0; k < n; ++k) {
        int rc = sg_pack_size(g, 1, &lo[(size_t)k * D], &hi[(size_t)k * D], nprop, props, 8, &bytes[k]);
        if (rc) return rc;
        tot += bytes[k];
    }
    DevBuf &cb = g->scratch[3];
    int rc = ensure(g->pool, cb, (size_t)tot + 64);
    if (rc) return rc;
    rc = sg_pack(g, n, lo.data(), hi.data(), nprop, props, 8, cb.p, tot, SG_MEM_DEVICE);
    if (rc) return rc;
    SG_HIP(hipStreamSynchronize(g->stream));  // the destinations read it on their streams
    int64_t at = 0;
    for (int k = 0; k < n; ++k) {
        int64_t used = 0;
        rc = sg_unpack(g->copies[k].dst, (const unsigned char *)cb.p + at, tot - at, SG_MEM_DEVICE,
                       g->copies[k].dst_lo, nprop, props, 8, &used);
        if (rc) return rc;
        at += used;
    }
    g->copies.clear();
    return SG_OK;
}

}  // namespace

extern "C" {

int sg_remove_add_unpack_finalize(sg_grid *g, int nprop, const int32_t *props)
{
    if (!g) return fail(SG_E_ARG, "null argument");
    int rc = check_props(g, nprop, props);
    if (rc) return rc;
    if ((rc = remove_queued_boxes(g))) return rc;
    return flush_unpacked(g, nprop, props);
}

int sg_copy_to(sg_grid *dst, sg_grid *src, const int32_t *src_lo, const int32_t *src_hi, const int32_t *dst_lo)
{
    if (!dst || !src || !src_lo || !src_hi || !dst_lo) return fail(SG_E_ARG, "null argument");
    if (dst->dim != src->dim) return fail(SG_E_ARG, "copy_to: grids of different dimension");
    sg_grid::copy_section c{};
    c.dst = dst;
    for (int d = 0; d < 3; ++d) {
        c.lo[d] = d < src->dim ? src_lo[d] : 0;
        c.hi[d] = d < src->dim ? src_hi[d] : 0;
        c.dst_lo[d] = d < src->dim ? dst_lo[d] : 0;
    }
    src->copies.push_back(c);
    return SG_OK;
}

int sg_remove_copy_to_finalize(sg_grid *g, int phase, int nprop, const int32_t *props)
{
    if (!g) return fail(SG_E_ARG, "null argument");
    int rc = check_props(g, nprop, props);
    if (rc) return rc;
    switch (phase & 3) {
    case SG_COPY_PHASE1: return remove_queued_boxes(g);
    case SG_COPY_PHASE2: return copy_sections_out(g, nprop, props);
    case SG_COPY_PHASE3: return flush_unpacked(g, nprop, props);
    default: return fail(SG_E_ARG, "bad phase");
    }
}

int sg_remove_add_unpack_reset(sg_grid *g)
{
    if (!g) return fail(SG_E_ARG, "null grid");
    g->rem_lo.clear();
    g->rem_hi.clear();
    g->copies.clear();
    g->ins_n = 0;
    g->cins_n = 0;
    g->pins_n = 0;
    return SG_OK;
}

}  // extern "C"
