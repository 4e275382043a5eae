// k_build.hip -- neighbour rebuild on gfx950: bounding box, Morton keys of
// the binning grid, permutation of the particle store, cell ranges, the
// Verlet list and the per-particle bond lists.
//
// Replaces, for the hot loop, the reference's Voronoi/k-d machinery
// (src/voronoi.h:77-237, src/kdtree.h:116-285, src/reorder.h:30-149,
// src/reorder_morton.h:44-122): particles are kept in Morton order of a
// uniform grid (cell edge >= lipid cutoff + skin), every particle lists all
// partners within rc(ti,tj) + skin, so the force kernel sees every pair the
// cutoff admits (the reference's centroid stencil can miss some; the
// Voronoi filter below reproduces its set when asked to).
#include <algorithm>

#include "orbc_internal.h"

namespace orbc {

namespace {

__device__ inline float normsq_unfused(float a, float b, float c) {
    return __fadd_rn(__fadd_rn(__fmul_rn(a, a), __fmul_rn(b, b)), __fmul_rn(c, c));
}

__global__ __launch_bounds__(BLOCK) void k_bbox_partial(const double *x, long long n, double *partial) {
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    for (long long i = (long long)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (long long)gridDim.x * BLOCK) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const double v = x[3 * i + d];
            lo[d] = fmin(lo[d], v);
            hi[d] = fmax(hi[d], v);
        }
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        for (int off = 32; off > 0; off >>= 1) {
            lo[d] = fmin(lo[d], __shfl_xor(lo[d], off, 64));
            hi[d] = fmax(hi[d], __shfl_xor(hi[d], off, 64));
        }
    }
    __shared__ double s[BLOCK / 64][6];
    const int wave = threadIdx.x >> 6;
    if (__lane_id() == 0)
        for (int d = 0; d < 3; ++d) { s[wave][d] = lo[d]; s[wave][3 + d] = hi[d]; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < BLOCK / 64; ++w)
            for (int d = 0; d < 3; ++d) {
                s[0][d] = fmin(s[0][d], s[w][d]);
                s[0][3 + d] = fmax(s[0][3 + d], s[w][3 + d]);
            }
        for (int d = 0; d < 6; ++d) partial[6 * blockIdx.x + d] = s[0][d];
    }
}

struct WrapArgs {
    double lo[3], L[3];
    int per[3];
};
__global__ __launch_bounds__(BLOCK) void k_wrap(double *x, long long n, WrapArgs w) {
    const long long i = (long long)blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n) return;
    for (int d = 0; d < 3; ++d)
        if (w.per[d]) {
            const double u = x[3 * i + d] - w.lo[d];
            x[3 * i + d] = w.lo[d] + (u - w.L[d] * floor(u / w.L[d]));
        }
}

// one wavefront: lanes stride over the block partials, then a shuffle reduction
__global__ void k_bbox_final(const double *partial, int nb, double *out) {
    double r[6] = {1e300, 1e300, 1e300, -1e300, -1e300, -1e300};
    for (int b = threadIdx.x; b < nb; b += 64)
        for (int d = 0; d < 3; ++d) {
            r[d] = fmin(r[d], partial[6 * b + d]);
            r[3 + d] = fmax(r[3 + d], partial[6 * b + 3 + d]);
        }
    for (int off = 32; off > 0; off >>= 1)
        for (int d = 0; d < 3; ++d) {
            r[d] = fmin(r[d], __shfl_xor(r[d], off, 64));
            r[3 + d] = fmax(r[3 + d], __shfl_xor(r[3 + d], off, 64));
        }
    if (threadIdx.x == 0)
        for (int d = 0; d < 6; ++d) out[d] = r[d];
}

__device__ inline int cell_coord(double v, double lo, double cs, int dim) {
    int c = (int)floor((v - lo) / cs);
    return c < 0 ? 0 : (c >= dim ? dim - 1 : c);
}

__device__ inline uint32_t morton_var(int cx, int cy, int cz, int bx, int by, int bz) {
    uint32_t key = 0;
    int pos = 0;
    const int mb = max(bx, max(by, bz));
    for (int b = 0; b < mb; ++b) {
        if (b < bx) key |= (uint32_t)((cx >> b) & 1) << pos++;
        if (b < by) key |= (uint32_t)((cy >> b) & 1) << pos++;
        if (b < bz) key |= (uint32_t)((cz >> b) & 1) << pos++;
    }
    return key;
}

// sort keys, and what the rest of the rebuild counts on: empty cell ranges, zero counters and step flags
__global__ __launch_bounds__(BLOCK) void k_keys(const double *x, long long n, Grid g, uint32_t *keys, uint32_t *vals,
                                                uint2 *crange, BuildFlags f) {
    const long long i = (long long)blockIdx.x * BLOCK + threadIdx.x;
    for (long long c = i; c < g.ncell; c += (long long)gridDim.x * BLOCK) crange[c] = make_uint2(0u, 0u);
    if (i == 0) f.clear();
    if (i >= n) return;
    const int cx = cell_coord(x[3 * i], g.lo[0], g.csd[0], g.dim[0]);
    const int cy = cell_coord(x[3 * i + 1], g.lo[1], g.csd[1], g.dim[1]);
    const int cz = cell_coord(x[3 * i + 2], g.lo[2], g.csd[2], g.dim[2]);
    keys[i] = morton_var(cx, cy, cz, g.bits[0], g.bits[1], g.bits[2]);
    vals[i] = (uint32_t)i;
}
__global__ void k_clear_flags(BuildFlags f) { f.clear(); }

// AoS triples: one thread per component, so three consecutive threads read
// one particle's triple and every store instruction writes a contiguous run
__global__ __launch_bounds__(BLOCK) void k_permute3(PermuteArgs a) {
    const long long e = (long long)blockIdx.x * BLOCK + threadIdx.x;
    if (e >= 3 * a.n) return;
    const long long i = e / 3;
    const long long src = 3 * (long long)a.perm[i] + (e - 3 * i);
    for (int k = 0; k < a.n3; ++k) a.dst3[k][e] = a.src3[k][src];
    for (int k = 0; k < a.nf3; ++k) a.dstf3[k][e] = a.srcf3[k][src];
}

// per-particle fields
__global__ __launch_bounds__(BLOCK) void k_permute(PermuteArgs a) {
    const long long i = (long long)blockIdx.x * BLOCK + threadIdx.x;
    if (i >= a.n) return;
    const long long p = a.perm[i];
    a.type_dst[i] = a.type_src[p];
    a.id_dst[i] = a.id_src[p];
    a.slot_dst[i] = a.slot_src[p];
    if (a.aff_src) a.aff_dst[i] = a.aff_src[p];
    if (a.grp_src) a.grp_dst[i] = a.grp_src[p];
    for (int k = 0; k < a.n1; ++k) a.dst1[k][i] = a.src1[k][p];
}

// ---- removal of particles (stray-lipid cleanup) -------------------------------
// flag[slot] = 1 for the deleted particles (flag zeroed on entry); keep[i] = !del[i]
__global__ __launch_bounds__(BLOCK) void k_del_flags(long long n, const uint32_t *slot, const uint32_t *del,
                                                     uint32_t *flag, uint32_t *keep) {
    const long long i = (long long)blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n) return;
    if (del[i]) flag[slot[i]] = 1u;
    keep[i] = del[i] ? 0u : 1u;
}

// kept particle i goes to pos[i]; its slot, if below pslot0 (a lipid), closes
// the gaps of the deleted slots below it (slot_pre: exclusive scan of flag)
__global__ __launch_bounds__(BLOCK) void k_compact(long long n, const uint32_t *del, const uint32_t *pos,
                                                   uint32_t *perm, uint32_t *slot, const uint32_t *slot_pre,
                                                   uint32_t pslot0) {
    const long long i = (long long)blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n || del[i]) return;
    perm[pos[i]] = (uint32_t)i;
    const uint32_t sl = slot[i];
    if (sl < pslot0) slot[i] = sl - slot_pre[sl];
}

// FP32 mirror of one particle: integer anchor per axis, offset from it
__device__ inline uint32_t anchor_of(const Anchor &a, const double (&x)[3], float (&r)[3]) {
    long long A[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        long long q = (long long)floor((x[d] - a.lo[d]) / a.hd[d]) - a.A0[d];
        if (a.L[d] > 0) {
            // periodic axis: x is wrapped into the box; guard the last anchor against rounding
            const long long M = 1LL << a.width[d];
            q = q < 0 ? 0 : (q > M - 1 ? M - 1 : q);
        }
        A[d] = q;
        r[d] = __double2float_rn(x[d] - anchor_pos(a, d, q));
    }
    return (uint32_t)A[0] | ((uint32_t)A[1] << a.shy) | ((uint32_t)A[2] << a.shz);
}

__device__ inline PQ mirror_of(const float (&r)[3], uint32_t w, const double (&nrm)[3], int type) {
    PQ q;
    q.x = make_float4(r[0], r[1], r[2], __uint_as_float(w));
    q.n = make_float4(__double2float_rn(nrm[0]), __double2float_rn(nrm[1]), __double2float_rn(nrm[2]),
                      __int_as_float(type));
    return q;
}

__global__ __launch_bounds__(BLOCK) void k_refresh(long long n, const double *x, const double *nrm,
                                                   const uint8_t *type, Anchor a, PQ *pq, float *rb,
                                                   uint32_t *anc) {
    const long long i = (long long)blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n) return;
    const double xi[3] = {x[3 * i], x[3 * i + 1], x[3 * i + 2]};
    float r[3];
    const uint32_t w = anchor_of(a, xi, r);
    anc[i] = w;
    rb[3 * i] = r[0]; rb[3 * i + 1] = r[1]; rb[3 * i + 2] = r[2];
    if (pq) {
        const double ni[3] = {nrm[3 * i], nrm[3 * i + 1], nrm[3 * i + 2]};
        pq[i] = mirror_of(r, w, ni, (int)type[i]);
    }
}

// cells number at most 2^32 (the Morton grid's bits)
__device__ inline uint32_t cell_lin(int cx, int cy, int cz, const Grid &g) {
    return ((uint32_t)cz * (uint32_t)g.dim[1] + (uint32_t)cy) * (uint32_t)g.dim[0] + (uint32_t)cx;
}
// the three cell coordinates side by side in one word (their bits add up to at most 32)
__device__ inline uint32_t cell_pack(const Grid &g, int cx, int cy, int cz) {
    return (uint32_t)cx | (g.bits[1] ? (uint32_t)cy << g.bits[0] : 0u) |
           (g.bits[2] ? (uint32_t)cz << (g.bits[0] + g.bits[1]) : 0u);
}
__device__ inline void cell_unpack(const Grid &g, uint32_t w, int &cx, int &cy, int &cz) {
    auto field = [&](int sh, int nb) { return nb ? (int)((w >> sh) & (0xffffffffu >> (32 - nb))) : 0; };
    cx = field(0, g.bits[0]); cy = field(g.bits[0], g.bits[1]); cz = field(g.bits[0] + g.bits[1], g.bits[2]);
}

// cell coordinate c + dc along axis d: wraps on a periodic axis; false if it
// leaves an open axis
__device__ inline bool cell_step(const Grid &g, int d, int c, int dc, int &out) {
    int v = c + dc;
    if (g.per[d]) {
        v %= g.dim[d];
        if (v < 0) v += g.dim[d];
    } else if (v < 0 || v >= g.dim[d]) {
        return false;
    }
    out = v;
    return true;
}

// The particle store in its new order, and everything that follows from a
// particle's new place, in one pass over it: the gather through the sort's
// permutation, the inverse map, the FP32 mirror with its anchor and build-time
// offset, the particle's cell (packed) with its offset in the cell, and the
// cell ranges (where the sorted keys change).  Separate passes read x and n
// again and cost a launch each.
__global__ __launch_bounds__(BLOCK) void k_place(PlaceArgs a) {
    __shared__ double s_x[3 * BLOCK], s_n[3 * BLOCK];
    __shared__ uint32_t s_perm[BLOCK];
    const PermuteArgs &p = a.p;
    const long long i0 = (long long)blockIdx.x * BLOCK, i = i0 + threadIdx.x;
    if (blockIdx.x == 0 && threadIdx.x == 0) *a.anc_dev = a.anc_grid;
    const uint32_t src = i < p.n ? p.perm[i] : 0u;
    s_perm[threadIdx.x] = src;
    __syncthreads();
    // triples one component per thread (contiguous stores); x and n also to LDS
#pragma unroll
    for (int u = 0; u < 3; ++u) {
        const int e = u * BLOCK + (int)threadIdx.x, q = e / 3;
        if (i0 + q >= p.n) break;
        const long long from = 3 * (long long)s_perm[q] + (e - 3 * q), to = 3 * i0 + e;
        const double vx = p.src3[0][from], vn = p.src3[1][from];
        s_x[e] = vx; s_n[e] = vn;
        p.dst3[0][to] = vx; p.dst3[1][to] = vn;
        for (int k = 2; k < p.n3; ++k) p.dst3[k][to] = p.src3[k][from];
        for (int k = 0; k < p.nf3; ++k) p.dstf3[k][to] = p.srcf3[k][from];
    }
    __syncthreads();
    if (i >= p.n) return;
    const int type = p.type_src[src];
    p.type_dst[i] = (uint8_t)type;
    p.id_dst[i] = p.id_src[src];
    const uint32_t slot = p.slot_src[src];
    p.slot_dst[i] = slot;
    a.inv[slot] = (uint32_t)i;
    if (p.aff_src) p.aff_dst[i] = p.aff_src[src];
    if (p.grp_src) p.grp_dst[i] = p.grp_src[src];
    for (int k = 0; k < p.n1; ++k) p.dst1[k][i] = p.src1[k][src];
    const int t = (int)threadIdx.x;
    const double x[3] = {s_x[3 * t], s_x[3 * t + 1], s_x[3 * t + 2]};
    float r[3];
    const uint32_t w = anchor_of(a.anc_grid, x, r);
    a.anc[i] = w;
    a.rb[3 * i] = r[0]; a.rb[3 * i + 1] = r[1]; a.rb[3 * i + 2] = r[2];
    if (a.pq) {
        const double nrm[3] = {s_n[3 * t], s_n[3 * t + 1], s_n[3 * t + 2]};
        a.pq[i] = mirror_of(r, w, nrm, type);
    }
    const Grid &g = a.g;
    int c[3];
    float rel[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        c[d] = cell_coord(x[d], g.lo[d], g.csd[d], g.dim[d]);
        rel[d] = __double2float_rn(x[d] - (g.lo[d] + g.csd[d] * (double)c[d]));
    }
    a.crel[i] = make_float4(rel[0], rel[1], rel[2], __int_as_float(type));
    a.ccell[i] = cell_pack(g, c[0], c[1], c[2]);
    const uint32_t key = a.skey[i], cl = cell_lin(c[0], c[1], c[2], g);
    if (i == 0 || a.skey[i - 1] != key) a.crange[cl].x = (uint32_t)i;
    if (i + 1 == p.n || a.skey[i + 1] != key) a.crange[cl].y = (uint32_t)(i + 1);
}

// ---- Verlet list -------------------------------------------------------
// A wave builds the rows of `span` consecutive particles, one grid cell after
// the other.  The particles of a cell's 3x3x3 neighbourhood sit
// one per lane in registers (NL_CHUNKS times 64 at once); the cell's own
// particles, some seven, are gone through one by one, each broadcast to all
// lanes and tested against 64 candidates at a time, and the hits are appended
// in candidate order (cells x fastest, then by index) by their rank in the
// ballot.  Positions are offsets in the cell (k_place), so a test is three
// subtractions of numbers of a few cell edges (rounding < 1e-6; the list
// cutoffs carry a margin of 1e-4), without anchors and, with the image's
// shift in the cell offset, without a minimum image.
//
// The rows are collected in LDS and written the cell's columns side by side.
//
// What bounds it: instruction issue (VALU 66 % busy, 4 to 5 waves a SIMD) on
// the full RBC (3.2 M particles, 28 entries each): 286 M VALU instructions,
// 0.75 to 0.80 ms; and it writes 0.94 GB where the entries are 0.36.  The build
// that this replaced -- (particle, stripe) lanes over candidates staged in
// LDS, a list of the occupied cells -- issued 503 M and took 0.85 ms, besides
// the five kernels that made its list.  One thread per particle scanning its
// 27 cells takes 1.10 ms (the lanes' cells hold different numbers of
// particles).
__device__ inline bool stencil_accept(const NlistArgs &a, int ti, int tj, const float (&ci)[3], uint32_t j) {
    // reference stencil radii: pp 9, pl 8, ll 6 (src/compute_pairwise_fused.h:141-284)
    const int cb = a.aff[j];
    const float d2 = normsq_unfused(__fsub_rn(a.centroids[3 * cb], ci[0]), __fsub_rn(a.centroids[3 * cb + 1], ci[1]),
                                    __fsub_rn(a.centroids[3 * cb + 2], ci[2]));
    const int nl = (ti == 0) + (tj == 0);
    const float Rs = nl == 2 ? 6.0f : (nl == 1 ? 8.0f : 9.0f);
    return d2 < Rs * Rs;
}

__device__ inline void cell_centroid(const NlistArgs &a, long long i, float (&ci)[3]) {
    const int ca = a.aff[i];
    ci[0] = a.centroids[3 * ca]; ci[1] = a.centroids[3 * ca + 1]; ci[2] = a.centroids[3 * ca + 2];
}

constexpr int NL_CHUNKS = 4;                // 64-candidate chunks held in registers
constexpr int NL_CAND = 64 * NL_CHUNKS;
constexpr int NL_COLS = 16;                 // particles of a cell taken together
constexpr int NL_ROWS = 48;                 // entries of a row collected in LDS (later ones are stored one by one)
constexpr int NL_PITCH = NL_COLS + 1;       // LDS row pitch: a particle's entries lie in different banks

template <bool STENCIL>
__global__ __launch_bounds__(64) void k_nlist(NlistArgs a, int span) {
    __shared__ float s_cut2[36];
    __shared__ float4 s_shift[27];                    // offset of each of the 27 cells
    __shared__ uint2 s_cand[NL_CAND];     // candidate and its cell (of the 27)
    __shared__ uint32_t s_row[NL_ROWS * NL_PITCH];
    const Grid &g = a.g;
    if (threadIdx.x < 36) s_cut2[threadIdx.x] = a.tab.cut2[threadIdx.x];
    if (threadIdx.x < 27) {
        const int k = (int)threadIdx.x;
        s_shift[k] = make_float4((float)(k % 3 - 1) * (float)g.csd[0], (float)((k / 3) % 3 - 1) * (float)g.csd[1],
                                 (float)(k / 9 - 1) * (float)g.csd[2], 0.f);
    }
    wave_sync();
    // consecutive blocks on one XCD: their candidates and list lines share its L2
    const unsigned nbk = gridDim.x, q8 = nbk >> 3, rr = nbk & 7u, xcd = blockIdx.x & 7u, kk = blockIdx.x >> 3;
    const long long lb = (xcd < rr) ? (long long)xcd * (q8 + 1) + kk : (long long)rr * (q8 + 1) + (long long)(xcd - rr) * q8 + kk;
    const int lane = __lane_id();
    const long long i0 = lb * span;
    const long long il = i0 + lane;
    const bool in = lane < span && il < a.n;
    const uint32_t word = in ? a.ccell[il] : 0u;
    // where a cell, or the wave's part of it, begins
    unsigned long long heads = __ballot(in && (lane == 0 || a.ccell[il - 1] != word));
    // particle range of this lane's cell of the 27 around the cell that begins at head h
    const int ox = lane % 3 - 1, oy = (lane / 3) % 3 - 1, oz = lane / 9 - 1;
    auto range = [&](int h) {
        uint2 r = make_uint2(0u, 0u);
        int cx, cy, cz, xx, yy, zz;
        cell_unpack(g, (uint32_t)lane_of((int)word, h), cx, cy, cz);
        if (lane < 27 && cell_step(g, 0, cx, ox, xx) && cell_step(g, 1, cy, oy, yy) && cell_step(g, 2, cz, oz, zz))
            r = a.crange[cell_lin(xx, yy, zz, g)];
        return r;
    };
    int h = (int)__ffsll((long long)heads) - 1;
    uint2 r = range(h);
    if (in) {
        // what follows from the particle alone: the default budget, the bond list
        a.bud2[il] = 0.f;
        if (a.bnd) {
            const uint32_t s = a.slot[il], b0 = a.bstart[s], b1 = a.bstart[s + 1];
            for (uint32_t k = b0; k < b1; ++k)
                a.bnd[(long long)(k - b0) * a.stride + il] = a.inv[a.bpartner[k]] | ((uint32_t)a.btype[k] << 30);
            a.nbnd[il] = (uint8_t)(b1 - b0);
        }
    }
    while (heads) {
        heads &= heads - 1;
        const uint32_t p0 = (uint32_t)(i0 + h), st = r.x, cntc = r.y - r.x;
        // the wave's part of the cell's own range
        const uint32_t pe = (uint32_t)min((long long)(uint32_t)lane_of((int)r.y, 13), i0 + span);
        if (heads) {                                 // the next cell's ranges, read while this one is worked on
            h = (int)__ffsll((long long)heads) - 1;
            r = range(h);
        }
        const uint32_t inc = wave_scan_u32(cntc), before = inc - cntc;
        const uint32_t total = (uint32_t)lane_of((int)inc, 63);
        for (uint32_t pb = p0; pb < pe; pb += NL_COLS) {
            const int np = (int)min((uint32_t)NL_COLS, pe - pb);
            const float4 me = a.crel[min(pb + lane, pe - 1)];
            int cntv = 0;                            // lane p: entries of particle pb + p
            for (uint32_t seg = 0; seg < total; seg += NL_CAND) {
                if (pb == p0 || total > NL_CAND) {
                    // the candidates in order, cell by cell
                    wave_sync();
                    for (uint32_t u = 0; __ballot(u < cntc); ++u) {
                        const uint32_t t = before + u - seg;
                        if (u < cntc && t < (uint32_t)NL_CAND) s_cand[t] = make_uint2(st + u, (uint32_t)lane);
                    }
                    wave_sync();
                }
                float qx[NL_CHUNKS], qy[NL_CHUNKS], qz[NL_CHUNKS], q0[NL_CHUNKS];
                uint32_t qj[NL_CHUNKS];
                int qt[NL_CHUNKS];
#pragma unroll
                for (int q = 0; q < NL_CHUNKS; ++q) {
                    const uint32_t off = seg + 64u * q;
                    qx[q] = 1e18f; qy[q] = 0.f; qz[q] = 0.f; q0[q] = -1.f; qj[q] = 0u; qt[q] = 0;
                    if (off < total && off + lane < total) {
                        const uint2 cd = s_cand[64 * q + lane];
                        const float4 sh = s_shift[cd.y], cj = a.crel[cd.x];
                        qx[q] = cj.x + sh.x; qy[q] = cj.y + sh.y; qz[q] = cj.z + sh.z;
                        qj[q] = cd.x;
                        qt[q] = __float_as_int(cj.w);
                        q0[q] = s_cut2[qt[q]];
                    }
                }
                for (int p = 0; p < np; ++p) {
                    const float mx = lane_of(me.x, p), my = lane_of(me.y, p), mz = lane_of(me.z, p);
                    const int ti = lane_of(__float_as_int(me.w), p);
                    const uint32_t i = pb + (uint32_t)p;
                    int cnt = lane_of(cntv, p);
                    float ci[3] = {0.f, 0.f, 0.f};
                    if (STENCIL) cell_centroid(a, i, ci);
#pragma unroll
                    for (int q = 0; q < NL_CHUNKS; ++q) {
                        if (seg + 64u * q >= total) break;
                        const float dx = mx - qx[q], dy = my - qy[q], dz = mz - qz[q];
                        // a pair without interaction has a negative cutoff and never passes
                        const float cut2 = ti == 0 ? q0[q] : s_cut2[ti * NT + qt[q]];
                        bool hit = dx * dx + dy * dy + dz * dz < cut2 && qj[q] != i;
                        if (STENCIL && hit) hit = stencil_accept(a, ti, qt[q], ci, qj[q]);
                        const unsigned long long hm = __ballot(hit);
                        const int more = (int)__popcll(hm), pos = rank_in(hm);
                        if (cnt + more <= NL_ROWS) {             // wave-uniform
                            if (hit) s_row[pos * NL_PITCH + (cnt * NL_PITCH + p)] = qj[q];
                        } else if (hit) {
                            if (cnt + pos < NL_ROWS) s_row[(cnt + pos) * NL_PITCH + p] = qj[q];
                            else if (cnt + pos < a.kmax) a.nbr[list_base(i, a.kmax) + (cnt + pos) * BLOCK] = qj[q];
                        }
                        cnt += more;
                    }
                    cntv = lane == p ? cnt : cntv;
                }
            }
            // the collected rows, the particles side by side
            wave_sync();
            const int len = min(cntv, min(a.kmax, NL_ROWS)), wide = np > 8, per = wide ? 4 : 8;
            const int col = wide ? lane & 15 : lane & 7, mylen = col < np ? __shfl(len, col, 64) : 0;
            uint32_t *const out = a.nbr + list_base((long long)pb + col, a.kmax);
            for (int k = wide ? lane >> 4 : lane >> 3; __ballot(k < mylen); k += per)
                if (k < mylen) out[k * BLOCK] = s_row[k * NL_PITCH + col];
            if (lane < np) {
                const uint32_t i = pb + (uint32_t)lane;
                a.nnbr[i] = (uint32_t)min(cntv, a.kmax);
                if (cntv == 0 && a.tab.budget_rings[__float_as_int(me.w)] > 0) a.lone_list[atomicAdd(a.lone_count, 1u)] = i;
                if (cntv > a.kmax) atomicMax(a.max_count, (unsigned)cntv);
            }
        }
    }
}

// Outer shells (Chebyshev distance 2..R) of the particles whose type reaches
// past the first ring (band-3 / actin, the sigma-3.4 LJ pair: a few percent),
// appended to the k_nlist entries.  far_slots names them by upload slot (a
// particle's type never changes, so the host writes the list once; collecting
// them at every build costs same-address atomics or a scan); the waves of the
// grid take them in turn.  A wave scans for one particle: 64 cells at a time have their ranges prefix-summed across
// the lanes, their particles are staged in LDS relative to the particle's own
// cell and tested 64 per round, hits appended in candidate order.
constexpr int FAR_CAP = 256;         // candidates staged per wave per pass
__global__ __launch_bounds__(BLOCK) void k_nlist_far(NlistArgs a) {
    __shared__ float4 s_x[BLOCK / 64][FAR_CAP];
    __shared__ uint32_t s_j[BLOCK / 64][FAR_CAP];
    __shared__ uint32_t s_pref[BLOCK / 64][65];
    __shared__ uint32_t s_cst[BLOCK / 64][64];
    __shared__ float s_cut2[36];
    if (threadIdx.x < 36) s_cut2[threadIdx.x] = a.tab.cut2[threadIdx.x];
    __syncthreads();
    const int w = threadIdx.x >> 6, lane = __lane_id();
    const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const long long m = a.far_n;
    const long long nw = (long long)gridDim.x * (BLOCK / 64);
    const Grid &g = a.g;
    const float edge[3] = {(float)g.csd[0], (float)g.csd[1], (float)g.csd[2]};
    for (long long q = (long long)blockIdx.x * (BLOCK / 64) + w; q < m; q += nw) {
        const long long i = a.inv[a.far_slots[q]];         // wave-uniform
        const float4 me = a.crel[i];
        const int ti = __float_as_int(me.w);
        int cx, cy, cz, cnt = (int)a.nnbr[i];
        cell_unpack(g, a.ccell[i], cx, cy, cz);
        float ci[3] = {0.f, 0.f, 0.f};
        if (a.aff) cell_centroid(a, i, ci);
        const int R = a.tab.rings[ti], D = 2 * R + 1, ncube = D * D * D;
        for (int base = 0; base < ncube; base += 64) {
            const int k = base + lane;
            uint32_t st = 0, cntc = 0;
            if (k < ncube) {
                const int dx = k % D - R, dy = (k / D) % D - R, dz = k / (D * D) - R;
                int xx, yy, zz;
                if (max(abs(dx), max(abs(dy), abs(dz))) >= 2 && cell_step(g, 0, cx, dx, xx) && cell_step(g, 1, cy, dy, yy) &&
                    cell_step(g, 2, cz, dz, zz)) {
                    const uint2 r = a.crange[cell_lin(xx, yy, zz, g)];
                    st = r.x;
                    cntc = r.y - r.x;
                }
            }
            uint32_t inc = cntc;
            for (int off = 1; off < 64; off <<= 1) {
                const uint32_t y = __shfl_up(inc, off, 64);
                if (lane >= off) inc += y;
            }
            const uint32_t total = __shfl(inc, 63, 64);
            wave_sync();
            s_pref[w][lane + 1] = inc;
            s_cst[w][lane] = st;
            if (lane == 0) s_pref[w][0] = 0;
            wave_sync();
            for (uint32_t off = 0; off < total; off += FAR_CAP) {
                const uint32_t mm = min((uint32_t)FAR_CAP, total - off);
                wave_sync();
                for (uint32_t t = lane; t < mm; t += 64) {
                    const uint32_t gidx = off + t;
                    int lo = 0, hi = 64;                // largest k with pref[k] <= gidx
                    while (hi - lo > 1) {
                        const int mid = (lo + hi) >> 1;
                        if (s_pref[w][mid] <= gidx) lo = mid; else hi = mid;
                    }
                    const uint32_t j = s_cst[w][lo] + (gidx - s_pref[w][lo]);
                    const int kc = base + lo;
                    const float4 c = a.crel[j];
                    s_x[w][t] = make_float4(c.x + (float)(kc % D - R) * edge[0], c.y + (float)((kc / D) % D - R) * edge[1],
                                            c.z + (float)(kc / (D * D) - R) * edge[2], c.w);
                    s_j[w][t] = j;
                }
                wave_sync();
                for (uint32_t t0 = 0; t0 < mm; t0 += 64) {
                    const uint32_t t = t0 + lane;
                    bool hit = false;
                    uint32_t j = 0;
                    if (t < mm) {
                        const float4 c = s_x[w][t];
                        j = s_j[w][t];
                        const int tj = __float_as_int(c.w);
                        const float dx = me.x - c.x, dy = me.y - c.y, dz = me.z - c.z;
                        hit = dx * dx + dy * dy + dz * dz < s_cut2[ti * NT + tj];
                        if (a.aff && hit) hit = stencil_accept(a, ti, tj, ci, j);
                    }
                    const unsigned long long hm = __ballot(hit);
                    if (hit) {
                        const int pos = cnt + __popcll(hm & lt);
                        if (pos < a.kmax) a.nbr[list_base(i, a.kmax) + pos * BLOCK] = j;
                    }
                    cnt += __popcll(hm);
                }
            }
        }
        if (lane == 0) {
            a.nnbr[i] = (uint32_t)(cnt < a.kmax ? cnt : a.kmax);
            if (cnt > a.kmax) atomicMax(a.max_count, (unsigned)cnt);
        }
    }
}

// skin check: *spent is set where a particle moved past its budget since the
// last build (skin/2, or the one k_budget gave it; half2 = (skin/2)^2), from
// the FP64 state, as the skin check of the step kernels.  Only waves that find
// one write, so a valid list costs the reads alone: reducing the largest
// displacement instead puts an atomic on one address in the way of every
// wave that raises it, 27 us against 3.5 us on 225,000 particles.
__global__ __launch_bounds__(BLOCK) void k_disp(long long n, const double *x, const uint32_t *anc, const float *rb,
                                                Anchor g, const float *bud2, const uint32_t *nnbr, double half2,
                                                unsigned *spent) {
    const long long i = (long long)blockIdx.x * BLOCK + threadIdx.x;
    bool past = false;
    if (i < n) {
        const uint32_t w = anc[i];
        const long long A[3] = {(long long)(w & g.mx), (long long)((w >> g.shy) & g.my), (long long)(w >> g.shz)};
        float d2 = 0.f;
        for (int d = 0; d < 3; ++d) {
            const float e = __double2float_rn(x[3 * i + d] - anchor_pos(g, d, A[d])) - rb[3 * i + d];
            d2 += e * e;
        }
        past = !((double)d2 <= half2);               // also when d2 is not a number
        if (past && isfinite(d2) && bud2 && nnbr[i] == 0 && bud2[i] > 0.f) past = d2 > bud2[i];
    }
    const unsigned long long over = __ballot(past);
    if (over && __lane_id() == (int)__ffsll((long long)over) - 1) *spent = LIST_SPENT;
}

// ---- block halos ------------------------------------------------------------
// One workgroup per particle block b (particles i0 = b * BLOCK ...): the
// distinct list entries outside the block go into an LDS hash set, and the
// order in which they first arrive numbers them: ext[b * HALO_EXT_MAX + e] is
// entry e.  Then each particle's entries are rewritten as 16-bit entries: the
// local index (t < BLOCK: particle i0 + t; BLOCK + e: ext entry e) in bits
// 0-9 and the neighbour's type in bits 10-12, two per word, word m of the
// row at nbr16[list_base(column, words) + m * BLOCK] (the column of the lane order below), rows padded to whole groups of
// HALO_GROUP entries with the particle's own local index and type 0
// (distance 0: no contribution).  Which ext slot an entry gets depends on the order of
// the LDS atomics; the values staged at those slots, and so the forces, do
// not.  A block with more than ext_cap (the halo capacity less BLOCK) distinct
// entries is marked HALO_OVERFLOW.  Its threads look at s_over once a batch, so
// they may put in some more first, up to filling the set: probing ends after
// HALO_HASH slots at the latest, and an entry that finds no slot comes when s_cnt
// is far past ext_cap.  In a block that does not overflow the set is at most
// HALO_EXT_MAX / HALO_HASH full and every probe sequence ends soon.  (Stopping each
// thread at its first entry too many takes a test per entry: 311 -> 331 us on
// 12,657 blocks of which none overflows, 59 -> 69 us on 844 of which 832 do.)
constexpr int HALO_HASH = 4096;
constexpr unsigned HALO_FEW = 512;           // blocks up to which four threads share a row, not two
constexpr uint32_t HALO_EMPTY = 0xffffffffu;
static_assert(HALO_EXT_MAX <= HALO_HASH / 4, "halo hash set too small");
static_assert(HALO_CAP == BLOCK + HALO_EXT && HALO_CAP64 <= HALO_CAP && HALO_CAP <= HALO_CAP_WIDE && HALO_CAP_WIDE <= 1024, "10-bit halo indices");
static_assert(NT <= 8, "3-bit types in the halo entries");

__device__ inline uint32_t halo_hash(uint32_t j) { return (j * 2654435761u) >> (32 - 12); }   // 12 = log2(HALO_HASH)

//
// THREADS / BLOCK threads share a row, each taking batches of HB entries in turn:
// what bounds a block is the chain of list loads and LDS atomics of a row.  With
// 1, 2 and 4 threads a row: 3 blocks 28, 15.4 and 10.9 us, 57 blocks 35, 19.5 and
// 13.1, 888 blocks 46, 33.8 and 33.9, 12,522 blocks 438, 383 and 411.
template <int THREADS>
__global__ __launch_bounds__(THREADS) void k_halo(long long n, int kmax, int words, const uint32_t *nbr,
                                                  const uint32_t *nnbr, const uint8_t *type, uint32_t *ext,
                                                  uint32_t *ext_cnt, uint32_t *nbr16, uint32_t *hinfo, int ext_cap) {
    constexpr int PARTS = THREADS / BLOCK;
    __shared__ uint32_t s_key[HALO_HASH];
    __shared__ uint16_t s_val[HALO_HASH];
    __shared__ int s_nn[BLOCK], s_rank[BLOCK];
    __shared__ int s_cnt, s_over;
    const int t = (int)threadIdx.x % BLOCK, part = (int)threadIdx.x / BLOCK;
    const long long b = blockIdx.x, i0 = b * BLOCK, i = i0 + t;
    const int nn = i < n ? (int)nnbr[i] : 0;
    for (int h = threadIdx.x; h < HALO_HASH; h += THREADS) s_key[h] = HALO_EMPTY;
    if (threadIdx.x == 0) { s_cnt = 0; s_over = 0; }
    if (part == 0) {
        s_nn[t] = i < n ? nn : -1;
        s_rank[t] = 0;
    }
    __syncthreads();
    const uint32_t self = (uint32_t)i;
    uint32_t *ext_b = ext + b * HALO_EXT_MAX;
    const uint32_t *const row = nbr + list_base(i, kmax);
    // entries in batches of HB (the loads of a batch in flight together);
    // own-block entries and the padding (the particle itself) are skipped
    constexpr int HB = 8;
    for (int k0 = part * HB; k0 < nn; k0 += PARTS * HB) {
        uint32_t jb[HB];
#pragma unroll
        for (int u = 0; u < HB; ++u) jb[u] = (k0 + u < nn) ? row[(k0 + u) * BLOCK] : self;
        if (__hip_atomic_load(&s_over, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) break;
#pragma unroll
        for (int u = 0; u < HB; ++u) {
            const uint32_t j = jb[u];
            if ((unsigned long long)((long long)j - i0) < (unsigned long long)BLOCK) continue;
            uint32_t h = halo_hash(j);
            for (int probe = 0; probe < HALO_HASH; ++probe) {
                const uint32_t prev = atomicCAS(&s_key[h], HALO_EMPTY, j);
                if (prev == HALO_EMPTY) {
                    const int e = atomicAdd(&s_cnt, 1);
                    if (e < ext_cap) {
                        s_val[h] = (uint16_t)e;
                        ext_b[e] = j;
                    } else {
                        atomicExch(&s_over, 1);
                    }
                    break;
                }
                if (prev == j) break;
                h = (h + 1) & (HALO_HASH - 1);
            }
        }
    }
    // lane order of the step kernels: the block's particles by list length,
    // longest first (ties by position; positions past n last), so that each
    // wave walks rows of similar length.  Lane `r` of the block takes particle
    // i0 + (hinfo[i0 + r] & 255), whose row, hinfo[i0 + r] >> 8 entries, is written
    // to column i0 + r.
    const int mine = s_nn[t];
    int rank = 0;
    for (int u = part * (BLOCK / PARTS); u < (part + 1) * (BLOCK / PARTS); ++u) {
        const int v = s_nn[u];
        rank += (v > mine) || (v == mine && u < t);
    }
    if (PARTS > 1) atomicAdd(&s_rank[t], rank);
    __syncthreads();
    if (s_over) {
        if (threadIdx.x == 0) ext_cnt[b] = HALO_OVERFLOW;
        return;
    }
    if (threadIdx.x == 0) ext_cnt[b] = (uint32_t)s_cnt;
    if (PARTS > 1) rank = s_rank[t];
    if (part == 0) hinfo[i0 + rank] = (uint32_t)t | (uint32_t)nn << 8;
    if (i >= n) return;
    // column i0 + rank < n: active particles rank first
    uint32_t *const row16 = nbr16 + list_base(i0 + rank, words);
    // local indices, HB entries (HB / 2 words) per batch; the row's words
    // [0, halo_row_words(nn)) are written, entries past nn being the particle
    // itself, and nn <= kmax keeps them inside halo_words(kmax)
    const int nw = halo_row_words(nn);
    for (int m0 = part * (HB / 2); m0 < nw; m0 += PARTS * (HB / 2)) {
        uint32_t jb[HB], tb[HB];
#pragma unroll
        for (int u = 0; u < HB; ++u) jb[u] = (m0 * 2 + u < nn) ? row[(m0 * 2 + u) * BLOCK] : self;
#pragma unroll
        for (int u = 0; u < HB; ++u) tb[u] = (m0 * 2 + u < nn) ? (uint32_t)type[jb[u]] : 0u;
#pragma unroll
        for (int q = 0; q < HB / 2; ++q) {
            if (m0 + q >= nw) break;
            uint32_t word = 0;
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) {
                const uint32_t j = jb[2 * q + hh];
                const long long d = (long long)j - i0;
                uint32_t l = (uint32_t)t;
                if (d >= 0 && d < BLOCK) {
                    l = (uint32_t)d;
                } else {
                    // j is in the set (no overflow): the probe ends at its slot
                    uint32_t h = halo_hash(j);
                    for (int probe = 0; probe < HALO_HASH; ++probe) {
                        if (s_key[h] == j) { l = (uint32_t)BLOCK + s_val[h]; break; }
                        h = (h + 1) & (HALO_HASH - 1);
                    }
                }
                word |= (l | (tb[2 * q + hh] << 10)) << (16 * hh);
            }
            row16[(m0 + q) * BLOCK] = word;
        }
    }
}

// Skin budget of isolated particles.  The list stays valid while every pair
// not in it keeps d_i + d_j < r_ij(build) - rc_ij.  A particle with list
// entries gets the usual budget skin/2 (its unlisted pairs start at rc + skin
// or more).  A particle with no entries at all (a lipid ejected from a
// vesicle, drifting away) gets b_i = min_j (r_ij - rc_ij) / 2 over the
// particles j it could interact with in the cells within R rings, capped by
// (R h - max_j rc_ij) / 2 for everything beyond them (h the shortest cell
// edge; a particle outside the cube of R rings is at least R h away): then any
// two particles keep d_i + d_j <= r_ij - rc_ij as long as each stays within
// its own budget.  R is the type's ring count; when that finds nothing closer
// than its cap and few particles are isolated, the cube is widened to
// BUDGET_FAR_RINGS, so a lipid flying off at several cutoffs per ten steps
// keeps the list for tens of steps instead of two.  Every isolated particle
// of one build uses the same widening (it depends only on their count), which
// keeps the pairwise argument above.  Stores b_i^2 (FP32, minus a rounding
// margin) where it exceeds (skin/2)^2, else 0 ("skin/2").  Open boxes only
// (the caller skips periodic ones).
constexpr int BUDGET_FAR_RINGS = 12;
constexpr long long BUDGET_FAR_MAX = 512;   // isolated particles for which the cube is widened
constexpr unsigned BUDGET_GRID = 512;       // blocks of k_budget

struct BudgetSite {
    double x, y, z, cmax;
    int ti, cx, cy, cz;
};

__device__ inline BudgetSite budget_site(long long i, const double *x, const uint8_t *type, const Grid &g,
                                         const ListTab &tab) {
    BudgetSite b;
    b.x = x[3 * i]; b.y = x[3 * i + 1]; b.z = x[3 * i + 2];
    b.ti = type[i];
    b.cmax = 0.0;
    for (int tj = 0; tj < NT; ++tj) b.cmax = fmax(b.cmax, (double)tab.pair_cut[b.ti * NT + tj]);
    b.cx = cell_coord(b.x, g.lo[0], g.csd[0], g.dim[0]);
    b.cy = cell_coord(b.y, g.lo[1], g.csd[1], g.dim[1]);
    b.cz = cell_coord(b.z, g.lo[2], g.csd[2], g.dim[2]);
    return b;
}

// min over the particles j != i of the cells of the cube of R rings, those within
// `inner` rings left out, of (r_ij - rc_ij) / 2; this thread takes the cells
// first, first + step, ...  The ranges of BUDGET_CELLS cells, then BUDGET_GROUP
// particles of a cell, are read together: one after the other each is a wait for
// memory (with 1024 threads a particle instead of 256: 91 -> 30 us for one lipid
// off a 14,000-particle vesicle, which the 25^3 cells hold whole).
constexpr int BUDGET_CELLS = 4, BUDGET_GROUP = 4, BUDGET_THREADS = 1024;
__device__ inline double budget_cells(long long i, const BudgetSite &b, int first, int step, int R, int inner,
                                      const double *x, const uint8_t *type, const Grid &g, const uint2 *crange,
                                      const ListTab &tab, double best) {
    const int side = 2 * R + 1, cells = side * side * side;
    for (int q0 = first; q0 < cells; q0 += BUDGET_CELLS * step) {
        uint2 cr[BUDGET_CELLS];
#pragma unroll
        for (int u = 0; u < BUDGET_CELLS; ++u) {
            const int q = q0 + u * step;
            const int dx = q % side - R, dy = (q / side) % side - R, dz = q / (side * side) - R;
            int xx, yy, zz;
            cr[u] = make_uint2(0u, 0u);
            if (q < cells && max(abs(dx), max(abs(dy), abs(dz))) > inner && cell_step(g, 0, b.cx, dx, xx) &&
                cell_step(g, 1, b.cy, dy, yy) && cell_step(g, 2, b.cz, dz, zz))
                cr[u] = crange[cell_lin(xx, yy, zz, g)];
        }
#pragma unroll
        for (int u = 0; u < BUDGET_CELLS; ++u) {
            for (uint32_t j0 = cr[u].x; j0 < cr[u].y; j0 += BUDGET_GROUP) {
                double d[BUDGET_GROUP][3];
                int t[BUDGET_GROUP];
#pragma unroll
                for (int v = 0; v < BUDGET_GROUP; ++v) {
                    const long long j = min(j0 + v, cr[u].y - 1);
                    for (int k = 0; k < 3; ++k) d[v][k] = x[3 * j + k];
                    t[v] = type[j];
                }
#pragma unroll
                for (int v = 0; v < BUDGET_GROUP; ++v) {
                    const double c = tab.pair_cut[b.ti * NT + t[v]];
                    if (j0 + v >= cr[u].y || j0 + v == (uint32_t)i || !(c > 0.0)) continue;
                    const double ex = b.x - d[v][0], ey = b.y - d[v][1], ez = b.z - d[v][2];
                    best = fmin(best, 0.5 * (sqrt(ex * ex + ey * ey + ez * ez) - c));
                }
            }
        }
    }
    return best;
}

__device__ inline double block_min(double v, double *s_red) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmin(v, __shfl_xor(v, off, 64));
    if (__lane_id() == 0) s_red[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = s_red[0];
    for (int w = 1; w < BUDGET_THREADS / 64; ++w) r = fmin(r, s_red[w]);
    __syncthreads();
    return r;
}

// list[0, *count): the isolated particles (appended by k_nlist).  Few: one block per particle, the cube of its type's rings and, if
// nothing there is closer than that cube's cap, the cube of BUDGET_FAR_RINGS.
// Many: one thread per particle over its type's rings.
__global__ __launch_bounds__(BUDGET_THREADS) void k_budget(const double *x, const uint8_t *type, Grid g, const uint2 *crange,
                                                  const uint32_t *list, const uint32_t *count, ListTab tab,
                                                  float half_skin, float *bud2) {
    __shared__ double s_red[BUDGET_THREADS / 64];
    const long long m = *count;
    const double h = fmin(g.csd[0], fmin(g.csd[1], g.csd[2]));
    if (m > BUDGET_FAR_MAX) {
        for (long long q = (long long)blockIdx.x * BUDGET_THREADS + threadIdx.x; q < m; q += (long long)gridDim.x * BUDGET_THREADS) {
            const long long i = list[q];
            const BudgetSite b = budget_site(i, x, type, g, tab);
            const int R = tab.budget_rings[b.ti];
            const double best = budget_cells(i, b, 0, 1, R, -1, x, type, g, crange, tab, 0.5 * (R * h - b.cmax));
            const float r = (float)best - 1e-4f;
            if (r > half_skin) bud2[i] = r * r;
        }
        return;
    }
    for (long long q = blockIdx.x; q < m; q += gridDim.x) {          // block-uniform
        const long long i = list[q];
        const BudgetSite b = budget_site(i, x, type, g, tab);
        const int R = tab.budget_rings[b.ti];
        double best = block_min(budget_cells(i, b, (int)threadIdx.x, BUDGET_THREADS, R, -1, x, type, g, crange, tab, 1e300), s_red);
        double cap = 0.5 * (R * h - b.cmax);
        if (best >= cap && BUDGET_FAR_RINGS > R) {
            // nothing within R rings limits the budget: the cells between R and
            // BUDGET_FAR_RINGS rings
            const double far = budget_cells(i, b, (int)threadIdx.x, BUDGET_THREADS, BUDGET_FAR_RINGS, R, x, type, g, crange, tab, 1e300);
            best = fmin(best, block_min(far, s_red));
            cap = 0.5 * (BUDGET_FAR_RINGS * h - b.cmax);
        }
        const float r = (float)fmin(best, cap) - 1e-4f;
        if (threadIdx.x == 0 && r > half_skin) bud2[i] = r * r;
    }
}

inline unsigned nblk(long long n) { return (unsigned)((n + BLOCK - 1) / BLOCK); }

}  // namespace

void launch_budget(const NlistArgs &a, const double *x, const uint8_t *type, float half_skin, hipStream_t s) {
    if (a.n <= 0) return;
    hipLaunchKernelGGL(k_budget, dim3((unsigned)std::min<long long>(nblk(a.n), BUDGET_GRID)), dim3(BUDGET_THREADS), 0, s, x, type,
                       a.g, a.crange, a.lone_list, a.lone_count, a.tab, half_skin, a.bud2);
}

void launch_halo(long long n, int kmax, const uint32_t *nbr, const uint32_t *nnbr, const uint8_t *type,
                 uint32_t *ext, uint32_t *cnt, uint32_t *nbr16, uint32_t *hinfo, int cap, hipStream_t s) {
    if (n <= 0) return;
    const dim3 g(nblk(n));
    const int w = (int)halo_words(kmax), cap_ext = cap - BLOCK;
    if (g.x <= HALO_FEW)
        hipLaunchKernelGGL(k_halo<1024>, g, dim3(1024), 0, s, n, kmax, w, nbr, nnbr, type, ext, cnt, nbr16, hinfo, cap_ext);
    else
        hipLaunchKernelGGL(k_halo<512>, g, dim3(512), 0, s, n, kmax, w, nbr, nnbr, type, ext, cnt, nbr16, hinfo, cap_ext);
}

void launch_disp(long long n, const double *x, const uint32_t *anc, const float *rb, Anchor g, const float *bud2,
                 const uint32_t *nnbr, double half2, unsigned *spent, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_disp, dim3(nblk(n)), dim3(BLOCK), 0, s, n, x, anc, rb, g, bud2, nnbr, half2, spent);
}

void launch_wrap(double *x, long long n, const double lo[3], const double L[3], const int per[3], hipStream_t s) {
    if (n <= 0) return;
    WrapArgs w{};
    for (int d = 0; d < 3; ++d) { w.lo[d] = lo[d]; w.L[d] = L[d]; w.per[d] = per[d]; }
    hipLaunchKernelGGL(k_wrap, dim3(nblk(n)), dim3(BLOCK), 0, s, x, n, w);
}

void launch_bbox(const double *x, long long n, double *out6, hipStream_t s) {
    // out6 must have room for 6 * 257 doubles: partials then result
    const int nb = 256;
    double *partial = out6 + 6;
    hipLaunchKernelGGL(k_bbox_partial, dim3(nb), dim3(BLOCK), 0, s, x, n, partial);
    hipLaunchKernelGGL(k_bbox_final, dim3(1), dim3(64), 0, s, partial, nb, out6);
}

void launch_keys(const double *x, long long n, Grid g, uint32_t *keys, uint32_t *vals, uint2 *crange,
                 const BuildFlags &f, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_keys, dim3(nblk(n)), dim3(BLOCK), 0, s, x, n, g, keys, vals, crange, f);
}

void launch_clear_flags(const BuildFlags &f, hipStream_t s) {
    hipLaunchKernelGGL(k_clear_flags, dim3(1), dim3(1), 0, s, f);
}

void launch_place(const PlaceArgs &a, hipStream_t s) {
    if (a.p.n <= 0) return;
    hipLaunchKernelGGL(k_place, dim3(nblk(a.p.n)), dim3(BLOCK), 0, s, a);
}

void launch_permute(const PermuteArgs &a, hipStream_t s) {
    if (a.n <= 0) return;
    if (a.n3 > 0 || a.nf3 > 0) hipLaunchKernelGGL(k_permute3, dim3(nblk(3 * a.n)), dim3(BLOCK), 0, s, a);
    hipLaunchKernelGGL(k_permute, dim3(nblk(a.n)), dim3(BLOCK), 0, s, a);
}

void launch_compact(long long n, const uint32_t *del, uint32_t *slot, uint32_t pslot0, uint32_t *flag,
                    uint32_t *slot_pre, uint32_t *keep, uint32_t *pos, uint32_t *perm, void *scan_temp,
                    hipStream_t s) {
    if (n <= 0) return;
    launch_fill_u32(flag, 0u, n, s);
    hipLaunchKernelGGL(k_del_flags, dim3(nblk(n)), dim3(BLOCK), 0, s, n, slot, del, flag, keep);
    exclusive_scan_u32(flag, slot_pre, n, scan_temp, s);
    exclusive_scan_u32(keep, pos, n, scan_temp, s);
    hipLaunchKernelGGL(k_compact, dim3(nblk(n)), dim3(BLOCK), 0, s, n, del, pos, perm, slot, slot_pre, pslot0);
}

void launch_refresh(long long n, const double *x, const double *nrm, const uint8_t *type, Anchor a, PQ *pq,
                    float *rb, uint32_t *anc, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_refresh, dim3(nblk(n)), dim3(BLOCK), 0, s, n, x, nrm, type, a, pq, rb, anc);
}

void launch_nlist(const NlistArgs &a, hipStream_t s) {
    if (a.n <= 0) return;
    // a wave's particles: 64 where that leaves every SIMD several waves, else
    // fewer, so that a small system's cells are built side by side
    const dim3 b(BLOCK);
    const int span = a.n >= 64 * 8192LL ? 64 : a.n >= 16 * 8192LL ? 16 : 8;
    const dim3 grid((unsigned)((a.n + span - 1) / span)), wave(64);
    if (a.aff) hipLaunchKernelGGL(k_nlist<true>, grid, wave, 0, s, a, span);
    else hipLaunchKernelGGL(k_nlist<false>, grid, wave, 0, s, a, span);
    if (a.far_n > 0) {
        // enough waves to fill the GPU; each takes list entries in turn
        const unsigned nb = (unsigned)std::min<long long>((a.far_n + BLOCK / 64 - 1) / (BLOCK / 64), 4096);
        hipLaunchKernelGGL(k_nlist_far, dim3(nb), b, 0, s, a);
    }
}

}  // namespace orbc
