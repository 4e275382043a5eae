// orbc_internal.h -- shared definitions of the gfx950 kernels and the host
// side of liborbc_hip.so.  Not part of the public ABI (include/orbc.h is).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <type_traits>

namespace orbc {

constexpr int NT = 6;     // particle types, src/forcefield_canonical.h:31-37
constexpr int NBT = 4;    // bond types, src/forcefield_canonical.h:101-109
constexpr int BLOCK = 256;
constexpr uint32_t BOND_INDEX_MASK = 0x3fffffffu;

// ---------------------------------------------------------------------------
// Force-field constants, src/forcefield_canonical.h:24-28,40-109.
// The lipid-lipid values are compile-time constants so the dominant pair type
// needs no table lookups; the tables are filled from the same expressions.
constexpr double kCutLL = 2.6, kReqLL = 1.1225, kEpsLL = 1.2, kAlphaLL = 1.55;
constexpr double ipow_c(double b, int e) { return e == 0 ? 1.0 : b * ipow_c(b, e - 1); }
constexpr double kRepLL = kEpsLL / ipow_c(kCutLL - kReqLL, 8);
constexpr double kAttLL = -2.0 * kEpsLL / ipow_c(kCutLL - kReqLL, 4);
constexpr double kCut2LL = kCutLL * kCutLL;

template <typename R>
struct FFTab {
    R cut2_poly[36], cut_poly[36], rep[36], att[36], alpha[36];
    R cut2_lj[36], lj1[36], lj2[36];
    int aniso[36];
    R mass[NT], inv_mass[NT];
    R bond_r0[NBT], bond_K[NBT];
};

void ff_fill(FFTab<double> &d, FFTab<float> &f);          // host, ff.cpp
double ff_max_cut(int a, int b);                            // rc(a,b), 0 if none

// ---------------------------------------------------------------------------
// Geometry of the FP32 mirrors: position = h * A + r, A an integer anchor per
// axis fixed at the last neighbour build, r the FP32 offset.  A - A0 is packed
// into 32 bits (bits[0] | bits[1] << shy | bits[2] << shz).
// Packed 32-bit integer anchor of each particle; the FP32 mirror stores the
// offset r = x - anchor position.  Per axis d the position of anchor A is
// lo[d] + hd[d] * (A + A0[d]).  Open axes: lo = 0 and hd a power of two, so
// hf * dA is exact in FP32.  Periodic axes: A0 = 0, lo = box origin,
// hd = L / 2^bits, and anchor differences wrap to the nearest image by sign
// extension from `bits` (width = bits; 31 on open axes, whose differences are
// less than 2^30: an axis has at most 30 bits).
struct Anchor {
    double hd[3];    // anchor spacing
    float hf[3];
    double lo[3];
    long long A0[3]; // anchor origin (open axes)
    unsigned shy, shz, mx, my, mz;
    unsigned nby;    // bits of the y field
    unsigned width[3];
    double L[3], Linv[3];   // periodic axes: box length (FP64 minimum image); 0 on open axes
};

struct AnchorI {
    int x, y, z;
};
__device__ inline AnchorI anchor_unpack(uint32_t w, const Anchor &a) {
    return AnchorI{(int)(w & a.mx), (int)__builtin_amdgcn_ubfe(w, a.shy, a.nby), (int)(w >> a.shz)};
}
// anchor difference to the nearest image (identity on open axes)
__device__ inline int anchor_wrap(int dA, unsigned width) { return __builtin_amdgcn_sbfe(dA, 0, width); }
// r + (distance between the anchors) with one rounding: on open axes the
// product is exact (power-of-two spacing), on periodic axes it is not
__device__ inline float anchor_add(const Anchor &a, int axis, float r, int dA) {
    return __fmaf_rn(a.hf[axis], (float)anchor_wrap(dA, a.width[axis]), r);
}
// the same separation in FP64 without rounding: the offsets differ exactly in
// FP64, and h * dA is exact on open axes (on periodic axes it carries the
// rounding of h = L / 2^bits only)
__device__ inline double anchor_add_exact(const Anchor &a, int axis, float ri, float rj, int dA) {
    return __fma_rn(a.hd[axis], (double)anchor_wrap(dA, a.width[axis]), (double)ri - (double)rj);
}
// FP64 position of anchor A along one axis
__device__ inline double anchor_pos(const Anchor &a, int axis, long long A) {
    return a.lo[axis] + a.hd[axis] * (double)(A + a.A0[axis]);
}
// FP64 minimum image on the periodic axes
__device__ inline void min_image(const Anchor &a, double &dx, double &dy, double &dz) {
    if (a.L[0] > 0) dx -= a.L[0] * rint(dx * a.Linv[0]);
    if (a.L[1] > 0) dy -= a.L[1] * rint(dy * a.Linv[1]);
    if (a.L[2] > 0) dz -= a.L[2] * rint(dz * a.Linv[2]);
}

// Uniform binning grid of the neighbour build (Morton-ordered cells).  On a
// periodic axis the cells tile [lo, lo + L) exactly and neighbour cells wrap.
struct Grid {
    double lo[3];
    double cs;       // nominal cell edge
    double csd[3];   // cell edge per axis (>= cs; L / dim on periodic axes)
    int dim[3];
    int bits[3];     // Morton bits per axis
    int per[3];      // periodic axis
    long long ncell;
};


// Skip gate for work launched ahead inside a batched run (orbc_run).  The
// work of step k is enqueued before step k's fused kernel; when *stop is set or
// step k-1 raised its skin flag (*slot), step k will be skipped, and every
// kernel of its work returns at once.  A default Gate is always open.
// Skip gate of the work queued before a batched step (see StepArgs::dslot):
// closed when the run has stopped or when the step's input positions violate
// the skin (slot (step + 2) % 3).  The step is *step0 + k when step0 is set
// (steps numbered on the device, so a captured graph serves any start step),
// else k.
struct Gate {
    const int *stop = nullptr;
    const unsigned *slots = nullptr;
    const unsigned long long *step0 = nullptr;
    unsigned long long k = 0;
};
__device__ inline bool gate_closed(const Gate &g) {
    if (!g.stop) return false;
    const unsigned long long st = (g.step0 ? *g.step0 : 0ull) + g.k;
    return *g.stop != 0 || g.slots[(st + 2ull) % 3ull] != 0u;
}

__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// inclusive sum over the wave by DPP moves (rows of 16, then across rows)
__device__ inline uint32_t wave_scan_u32(uint32_t x) {
    auto dpp = [](uint32_t v, auto ctrl, auto rows) {
        return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, decltype(ctrl)::value, decltype(rows)::value, 0xf, false);
    };
    using std::integral_constant;
    x += dpp(x, integral_constant<int, 0x111>{}, integral_constant<int, 0xf>{});   // row_shr:1
    x += dpp(x, integral_constant<int, 0x112>{}, integral_constant<int, 0xf>{});   // row_shr:2
    x += dpp(x, integral_constant<int, 0x114>{}, integral_constant<int, 0xf>{});   // row_shr:4
    x += dpp(x, integral_constant<int, 0x118>{}, integral_constant<int, 0xf>{});   // row_shr:8
    x += dpp(x, integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{});   // row_bcast:15 into rows 1, 3
    x += dpp(x, integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{});   // row_bcast:31 into rows 2, 3
    return x;
}
__device__ inline int lane_of(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ inline float lane_of(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
// bits of m below this lane
__device__ inline int rank_in(unsigned long long m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
// smallest value of the wave, in every lane
__device__ inline float wave_min(float x) {
    auto step = [&x](auto ctrl, auto rows) {
        const int v = __float_as_int(x);
        x = fminf(x, __int_as_float(__builtin_amdgcn_update_dpp(v, v, decltype(ctrl)::value, decltype(rows)::value, 0xf, false)));
    };
    using std::integral_constant;
    step(integral_constant<int, 0x111>{}, integral_constant<int, 0xf>{});
    step(integral_constant<int, 0x112>{}, integral_constant<int, 0xf>{});
    step(integral_constant<int, 0x114>{}, integral_constant<int, 0xf>{});
    step(integral_constant<int, 0x118>{}, integral_constant<int, 0xf>{});
    step(integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{});
    step(integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{});
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}

// FP32 mirror of one particle for the mixed path, one 32-byte record so a
// neighbour gather touches one cache line: x = position offset from the
// anchor (xyz) + packed anchor (w, bits); n = director (xyz) + type (w, bits).
struct PQ {
    float4 x, n;
};

// Block halos of the mixed step (k_halo, k_step_langevin): particle block b
// (the BLOCK particles from b * BLOCK in store order) stages its own mirrors
// and those of at most HALO_EXT distinct outside neighbours in LDS, and walks
// its list as 16-bit entries (10-bit index into that table, 3-bit type).  A block with more outside
// neighbours is marked HALO_OVERFLOW and gathers from the 32-bit list.
#ifndef ORBC_HALO_CAP
#define ORBC_HALO_CAP 896
#endif
constexpr int HALO_CAP = ORBC_HALO_CAP;        // local indices: BLOCK own + HALO_EXT outside (default)
constexpr int HALO_EXT = HALO_CAP - BLOCK;
// the default halos of FP64, whose records are 48 bytes: as many as leave a CU's
// LDS to four blocks (896 leave it to three: 398 us a launch on 3.2 M particles
// against 374 on average, although 37 of 12,522 blocks now overflow against 4)
#ifndef ORBC_HALO_CAP64
#define ORBC_HALO_CAP64 800
#endif
constexpr int HALO_CAP64 = ORBC_HALO_CAP64;
// the wide variant (the autotuner's halo capacity knob): 1024 local indices,
// the most the 10-bit index holds, at one block fewer per CU
constexpr int HALO_CAP_WIDE = 1024;
constexpr int HALO_EXT_MAX = HALO_CAP_WIDE - BLOCK;   // ext entries kept per block (array stride)
constexpr uint32_t HALO_OVERFLOW = 0xffffffffu;
// entries per group of the LDS walk (rows are padded to whole groups)
#ifndef ORBC_HALO_GROUP
#define ORBC_HALO_GROUP 4
#endif
constexpr int HALO_GROUP = ORBC_HALO_GROUP;
static_assert(HALO_GROUP == 4 || HALO_GROUP == 8, "halo group of 4 or 8 entries");
// 32-bit words of 16-bit entries in a row of nn entries (whole groups)
__host__ __device__ inline int halo_row_words(int nn) { return (HALO_GROUP / 2) * ((nn + HALO_GROUP - 1) / HALO_GROUP); }
inline long long halo_words(int kmax) { return halo_row_words(kmax); }

// Neighbour lists (32-bit entries, and the 16-bit ones of the block halos) are
// tiled by particle block: the k-th entries of a block's BLOCK particles lie
// side by side, its rows one after the other.  A block's list is then one
// contiguous piece (48 KB at 48 rows); with the k-th entries of all particles
// side by side a wave's rows lie n entries apart, each in a page of its own.
// Entry k of particle i is at list_base(i, rows) + k * BLOCK.
__host__ __device__ inline long long list_base(long long i, int rows) { return (i / BLOCK * rows) * BLOCK + i % BLOCK; }

// The thermostat's friction as a kernel of the batched Nose-Hoover run finds it:
// *in, or with nb > 0 what k_zeta_update makes of it from the nb kinetic-energy
// partials of the kernel before, in the same order of additions; the first block
// leaves it in *out for the kernel after.
constexpr int ZETA_PARTS = 1024;   // partials that a block adds up itself, at most
struct ZetaUp {
    const double *partial;
    int nb;
    const double *in;
    double *out;
    double dt, Q, nkT15;
};
// wave sums of the partials into ws[ZETA_PARTS / 64]: wave v holds partials 64 v ...; all BLOCK threads, before a barrier
__device__ inline void zeta_sums(const ZetaUp &z, double *ws) {
    const int lane = __lane_id(), wave = (int)threadIdx.x >> 6;
    double x[ZETA_PARTS / BLOCK];
#pragma unroll
    for (int j = 0; j < ZETA_PARTS / BLOCK; ++j) {
        const int k = j * BLOCK + (int)threadIdx.x;
        x[j] = k < z.nb ? z.partial[k] : 0.0;
    }
#pragma unroll
    for (int j = 0; j < ZETA_PARTS / BLOCK; ++j) {
        if (j * BLOCK >= z.nb) {
            if (lane == 0) ws[j * (BLOCK / 64) + wave] = 0.0;
            continue;
        }
        for (int off = 32; off > 0; off >>= 1) x[j] += __shfl_xor(x[j], off, 64);
        if (lane == 0) ws[j * (BLOCK / 64) + wave] = x[j];
    }
}
// after the barrier
__device__ inline double zeta_now(const ZetaUp &z, const double *ws) {
    double ke = 0;
    for (int w = 0; w < ZETA_PARTS / 64; ++w) ke += ws[w];
    const double zeta = __builtin_fma(0.5 * z.dt / z.Q, ke - z.nkT15, *z.in);
    if (blockIdx.x == 0 && threadIdx.x == 0) *z.out = zeta;
    return zeta;
}

// Everything a step kernel reads or writes, by value in kernel arguments.
struct StepArgs {
    long long n;
    long long stride;          // column stride of the bond lists (>= n)
    int kmax, words;           // rows of a block in nbr and in nbr16
    // FP64 state (x, n read from *_in and written to *_out; v, o in place)
    const double *x_in, *n_in;
    double *x_out, *n_out, *v, *o;
    // FP32 mirrors (mixed precision)
    const PQ *pq_in;
    PQ *pq_out;
    const uint8_t *type;
    const uint32_t *id;
    const uint32_t *anc;       // packed anchors (FP64 path)
    const float *rb;           // offsets at the last build (skin check)
    const uint32_t *nbr, *nnbr;
    // block halos (mixed path; null: every block gathers from nbr)
    const uint32_t *halo_ext, *halo_cnt, *nbr16;
    const uint32_t *hinfo;   // of lane r of a halo block (k_halo): the particle's place in the block, list length << 8
    int halo_cap;            // local indices of the halos (HALO_CAP, HALO_CAP64 in FP64, or HALO_CAP_WIDE)
    const uint32_t *bnd;
    const uint8_t *nbnd;
    int has_bonds;
    // volume push fused into the step (constrain_volume): f += *push * mass_type * normal[aff]
    const double *push;        // device scalar strength (V0 - V) / V0, or null
    // the same from up to 64 partial sums of V, added up by each block (or null)
    const double *vol_partial;
    int vol_parts;
    double vol_target, vol_strength;
    const double *cell_normal; // 3 per Voronoi cell
    const int32_t *aff;        // Voronoi cell of each particle
    Anchor anc_grid;
    double dt;
    double gamma[NT], sigma[NT];
    // ensemble members with their own temperature: sigma of particle i is
    // sig_group[grp[i] * NT + type]; null: sigma[type]
    const uint16_t *grp;
    const double *sig_group;
    unsigned long long seed, step;
    // step0 set: the step is *step0 + step (device-side numbering of a
    // captured batch); null: the step is `step`
    const unsigned long long *step0;
    // the anchor grid as the step kernels read it: a device copy of anc_grid,
    // rewritten at every neighbour rebuild (so captured batches stay valid)
    const Anchor *anc_dev;
    // skin criterion on the device: step k reads slot (k+2)%3 (displacement of
    // its input positions), writes slot k%3 (of its output) and clears slot
    // (k+1)%3 for step k+1.  A step whose input violates the skin, or that
    // finds *stop set, does nothing and sets *stop, so the host can launch a
    // batch of steps and rebuild once after it.
    unsigned *dslot;           // 3 flags: some particle moved more than skin/2 since build
    float half_skin2;          // (skin/2)^2
    const float *bud2;         // squared skin budget of isolated particles (k_budget; 0: skin/2), or null
    int *stop;                 // sticky: a step was skipped
    int *done;                 // steps executed (incremented by block 0)
    int nh_gate;               // Nose-Hoover second half in a batch: skip on *stop or dslot[step % 3]
    unsigned *bad;             // nonzero if a non-finite value appeared
    int swizzle;               // XCD-aware block remap
};

// A step of the minimiser: the state and lists as a step kernel has them, and
struct MinArgs {
    StepArgs s;
    double box_lo[3], box_hi[3];
    double dr_opt, dn_opt;     // largest move of a position and of a director
    double half2;              // (skin/2)^2
};

// Per-particle accumulators for the standalone force / bond / integrate API.
struct ForceArgs {
    long long n, stride;       // particles, column stride of the bond lists
    int kmax;                  // rows of a block in nbr
    const double *x, *nrm;
    const PQ *pq;
    const uint8_t *type;
    const uint32_t *id;
    const uint32_t *nbr, *nnbr;
    const uint32_t *bnd;
    const uint8_t *nbnd;
    Anchor anc_grid;
    float *f32, *t32;
    double *f64, *t64;
    double *e, *w;
    int swizzle;
};

// ---------------------------------------------------------------------------
// launchers (each .hip file owns its kernels)
void upload_ff(const FFTab<double> &d, const FFTab<float> &f, hipStream_t s);

// k_sort.hip
size_t scan_temp_bytes(long long n);
void exclusive_scan_u32(const uint32_t *in, uint32_t *out, long long n, void *temp, hipStream_t s, Gate gt = {});
size_t radix_temp_bytes(long long n);
// allocation-free sort (k_sort.hip): the device address of this device's
// fixed scratch (looked up once per device, with it current) and the sort of
// caller-owned device arrays through that scratch
constexpr long long NOALLOC_SORT_MAX = 1LL << 20;
void *scratch_address(int device);
void sort_pairs_in_scratch(uint32_t *keys, uint32_t *vals, long long n, int bits, void *scr, hipStream_t s);
void radix_sort_pairs(uint32_t *keys, uint32_t *vals, uint32_t *keys_alt, uint32_t *vals_alt, long long n,
                      int bits, void *temp, hipStream_t s, bool *result_in_alt, Gate gt = {});

// k_build.hip
void launch_bbox(const double *x, long long n, double *out6, hipStream_t s);
// periodic axes: x -> lo + (x - lo) - L floor((x - lo) / L)
void launch_wrap(double *x, long long n, const double lo[3], const double L[3], const int per[3], hipStream_t s);
// counters and flags a rebuild starts from: the list counters, the largest
// displacement since the build, the skin flags of the batched steps and the
// stop flag
struct BuildFlags {
    unsigned *disp, *slots, *max_count, *lone_count;
    int *stop;
    __device__ void clear() const {
        *disp = 0u; *max_count = 0u; *lone_count = 0u;
        slots[0] = slots[1] = slots[2] = 0u;
        *stop = 0;
    }
};
void launch_keys(const double *x, long long n, Grid g, uint32_t *keys, uint32_t *vals, uint2 *crange,
                 const BuildFlags &f, hipStream_t s);
void launch_clear_flags(const BuildFlags &f, hipStream_t s);
struct PermuteArgs {
    long long n;
    const uint32_t *perm;
    const double *src3[6]; double *dst3[6]; int n3;     // AoS double3 arrays
    const float *srcf3[2]; float *dstf3[2]; int nf3;    // AoS float3 arrays
    const uint8_t *type_src; uint8_t *type_dst;
    const uint32_t *id_src; uint32_t *id_dst;
    const uint32_t *slot_src; uint32_t *slot_dst;
    const int32_t *aff_src; int32_t *aff_dst;
    const uint16_t *grp_src; uint16_t *grp_dst;         // ensemble member (or null)
    const double *src1[2]; double *dst1[2]; int n1;     // one number per particle
};
void launch_permute(const PermuteArgs &a, hipStream_t s);
// a permutation by sorted cell and all that depends on a particle's new place (k_place)
struct PlaceArgs {
    PermuteArgs p;             // src3/dst3 [0] and [1]: positions and directors
    Grid g;
    Anchor anc_grid;
    Anchor *anc_dev;           // device copy of anc_grid
    const uint32_t *skey;      // sorted cell keys
    uint32_t *inv;             // slot -> particle
    PQ *pq;                    // or null (FP64)
    float *rb;
    uint32_t *anc;
    float4 *crel;              // offset from the cell's corner, type
    uint32_t *ccell;           // packed cell coordinates
    uint2 *crange;             // [first, last) particle of every cell
};
void launch_place(const PlaceArgs &a, hipStream_t s);
// removal of the particles with del[i] != 0: perm[0..n - ndel) lists the kept
// particles in store order; lipid slots (< pslot0) are renumbered without
// gaps (flag, slot_pre, keep, pos: n-entry scratch)
void launch_compact(long long n, const uint32_t *del, uint32_t *slot, uint32_t pslot0, uint32_t *flag,
                    uint32_t *slot_pre, uint32_t *keep, uint32_t *pos, uint32_t *perm, void *scan_temp,
                    hipStream_t s);
void launch_refresh(long long n, const double *x, const double *nrm, const uint8_t *type, Anchor a,
                    PQ *pq, float *rb, uint32_t *anc, hipStream_t s);
// list cutoffs and search rings for a skin, per (type, type) or type
struct ListTab {
    float cut2[36];            // (rc(a,b) + skin)^2, < 0 if a, b never interact
    float pair_cut[36];        // interaction cutoff (0: none)
    int rings[NT];             // grid rings a type searches
    int budget_rings[NT];      // rings searched for the skin budget of an isolated particle (0: none)
};
struct NlistArgs {
    long long n, stride;
    const float4 *crel;        // offset of each particle from its cell's corner (xyz), type (w, bits)
    const uint32_t *ccell;     // packed cell of each particle
    const uint2 *crange;       // [first, last) particle of every grid cell
    Grid g;
    ListTab tab;
    uint32_t *nbr, *nnbr;
    int kmax;
    unsigned *max_count;       // the longest row, where it exceeds kmax
    const uint32_t *far_slots; // upload slots of the particles that search past the first ring
    long long far_n;
    uint32_t *lone_list;       // particles without entries
    unsigned *lone_count;
    float *bud2;
    const uint32_t *inv;       // slot -> particle
    // bond lists of the new order (k_nlist's threads also write them), or bnd null
    const uint32_t *slot, *bstart, *bpartner;
    const uint8_t *btype;
    uint32_t *bnd;
    uint8_t *nbnd;
    const int32_t *aff;        // Voronoi filter (null in exact mode)
    const float *centroids;
};
void launch_nlist(const NlistArgs &a, hipStream_t s);
// skin budget of the particles without list entries (k_build.hip, k_budget)
void launch_budget(const NlistArgs &a, const double *x, const uint8_t *type, float half_skin, hipStream_t s);
// sets *spent to LIST_SPENT where a particle is past its budget; half2 = (skin/2)^2,
// bud2: skin budgets of the last build (nullptr: skin/2 for every particle)
constexpr unsigned LIST_SPENT = 0x7f000000u;    // as float bits: larger than any (skin/2)^2
void launch_disp(long long n, const double *x, const uint32_t *anc, const float *rb, Anchor g, const float *bud2,
                 const uint32_t *nnbr, double half2, unsigned *spent, hipStream_t s);
// block halos from the 32-bit list: ext (HALO_EXT per block), cnt (per block),
// nbr16 (halo_words(kmax) rows a block)
void launch_halo(long long n, int kmax, const uint32_t *nbr, const uint32_t *nnbr, const uint8_t *type,
                 uint32_t *ext, uint32_t *cnt, uint32_t *nbr16, uint32_t *hinfo, int cap, hipStream_t s);

// k_force.hip
void launch_forces(const ForceArgs &a, bool mixed, bool energy, bool pair, bool bond, hipStream_t s);
void launch_step_langevin(const StepArgs &a, bool mixed, hipStream_t s);
// forces + the NH second half in one pass (k_forces + post_toque_final_update);
// f, n x t go to f32/t32 (mixed) or f64/t64, KE partials per particle block
void launch_step_nh_second(const StepArgs &a, bool mixed, float *f32, float *t32, double *f64, double *t64,
                           double *ke_partial, const ZetaUp &zeta, hipStream_t s);
// minimiser: forces, torque, capped descent step, walls and skin check of one step in one pass
void launch_min_step(const MinArgs &a, bool mixed, hipStream_t s);
void launch_pairs_export(const ForceArgs &a, bool mixed, unsigned *ids_i, unsigned *ids_j,
                         unsigned long long *count, long long cap, hipStream_t s);

// k_integrate.hip
struct IntegArgs {
    long long n;
    double *x, *v, *nrm, *o;
    float *f32, *t32;
    double *f64, *t64;
    const uint8_t *type;
    const uint32_t *id;
    const uint32_t *anc;
    PQ *pq;            // mirrors refreshed in place when nonnull
    Anchor anc_grid;
    double dt;
    double gamma[NT], sigma[NT];
    const uint16_t *grp;      // ensemble member of each particle, or null (see StepArgs)
    const double *sig_group;
    unsigned long long seed, step;
    double box_lo[3], box_hi[3];
    const double *zeta;       // device scalar
    ZetaUp zup;               // nb > 0: k_nh_first takes the friction from here
    double *ke_partial;       // per block
    // NH first half: when disp_max is set, the largest squared displacement of
    // the new positions from the build-time offsets rb (as k_disp computes it)
    // is folded into *disp_max (float bits, atomicMax)
    const float *rb;
    unsigned *disp_max;
    // batched Nose-Hoover run (orbc_run): stop set -> the kernel does nothing;
    // skin_slot set -> the first half ors 1 into it where a particle moved
    // past its budget (skin/2, or bud2 for particles without list entries) and
    // clears skin_clear for the step after
    const int *stop;
    unsigned *skin_slot, *skin_clear;
    const float *bud2;
    const uint32_t *nnbr;
    float half_skin2;
};
void launch_integrate(int kernel, const IntegArgs &a, bool mixed, hipStream_t s);
void launch_reduce_ke(const double *v, const uint8_t *type, long long n, double *partial, hipStream_t s);
void launch_sum_partials(const double *partial, long long nblocks, double *out, hipStream_t s);
void launch_zeta_update(const double *partial, long long nblocks, double *zeta, double dt, double Q,
                        double nkT15, hipStream_t s, const int *stop = nullptr, const double *zeta_in = nullptr);
void launch_sum_array(const double *a, long long n, double *partial, hipStream_t s);
long long reduce_blocks(long long n);
// up to four per-particle arrays of n < 2^30 particles into host arrays the
// GPU can write, in upload order (inv: slot -> particle, from the first slot)
struct ReadArgs {
    long long n;
    const uint32_t *inv;
    int nf;
    const void *src[4];
    double *dst[4];
    int width[4];              // numbers per particle: 3, or 1 (double only)
    int narrow[4];             // source is float
};
void launch_read(const ReadArgs &a, hipStream_t s);
void launch_scatter_slots(long long n, const uint32_t *slot, const double *src3, double *dst3, hipStream_t s);
void launch_scatter_slots_f(long long n, const uint32_t *slot, const float *src3, double *dst3, hipStream_t s);
void launch_scatter_slots1(long long n, const uint32_t *slot, const double *src, double *dst, hipStream_t s);
void launch_gather_slots(long long n, const uint32_t *slot, const double *src3, double *dst3, hipStream_t s);
void launch_gather_slots_f(long long n, const uint32_t *slot, const double *src3, float *dst3, hipStream_t s);
// before a batch of steps: no step done, and the device's step counter
void launch_batch_begin(int *done, unsigned long long *step, unsigned long long v, hipStream_t s);
// *p += v
void launch_add_u64(unsigned long long *p, unsigned long long v, hipStream_t s);
void launch_fill_u32(uint32_t *p, uint32_t v, long long n, hipStream_t s, Gate gt = {});
void launch_gather_u16(long long n, const uint32_t *slot, const uint16_t *src, uint16_t *dst, hipStream_t s);

// k_voronoi.hip
struct VoroArgs {
    long long n;            // particles
    long long ncell;
    const double *x;
    const double *nrm;
    const uint8_t *type;
    int32_t *aff;
    float *centroids;
    double mass[NT];
    // centroid grid (for nearest / within queries)
    Grid cg;
    const uint32_t *cg_start, *cg_end, *cg_idx;
    Gate gate;               // inside a batched run: the step this work precedes may be skipped
    const Grid *cg_dev;      // the centroid grid as the kernels read it: a device copy of cg, rewritten
                             // whenever the grid is rebuilt (so captured batches stay valid)
    // The centroid grid is built at neighbour rebuilds only: cref holds the
    // centroids as binned, *cdisp the largest squared drift of a centroid since
    // (as float bits).  Queries widen their reach by that drift, so they stay
    // exact.  cdisp null: the index is current.
    float *cref;
    unsigned *cdisp;
    // lipid count per cell of the current affiliation, written by
    // k_volume_finish; csize[ncell] != 0 says they are current (a partition
    // clears it).  A block of k_cell_sums holding every member of a cell
    // stores that cell's sums instead of adding them atomically.  Null: none.
    uint32_t *csize;
};
void launch_morton_ref(const float *pts, long long n, double bsize, uint32_t *keys, hipStream_t s);
// sort keys of m > 0 points, empty ranges (g.ncell of start and end) and, unless null, cref = c and *cdisp = 0
void launch_centroid_keys(const float *c, long long m, Grid g, uint32_t *keys, uint32_t *vals, uint32_t *start,
                          uint32_t *end, float *cref, unsigned *cdisp, hipStream_t s, Gate gt = {});
void launch_cgrid_ranges(const uint32_t *sorted_keys, long long ncell, uint32_t *start, uint32_t *end,
                         hipStream_t s, Gate gt = {});
// stray-lipid cleanup (src/cleanup.h:29-91)
void launch_stray_keys(const VoroArgs &a, uint32_t *keys, uint32_t *vals, double *d2, hipStream_t s);
void launch_stray_mark(long long ncell, const uint32_t *start, const uint32_t *end, const uint32_t *svals,
                       const double *d2, double tol2, uint32_t *del, unsigned *count, hipStream_t s);
void launch_nearest(const VoroArgs &a, const float *q, long long nq, const double *qd, int32_t *out, bool warm,
                    hipStream_t s);
void launch_within(const VoroArgs &a, const float *q, long long nq, float rmax, int cap, int *counts,
                   int *out, hipStream_t s);
void launch_centroid_sums(const VoroArgs &a, unsigned long long *sums, hipStream_t s);
// ... and the block sums of the new centroids, for the centre, to partial
void launch_centroid_finish(const VoroArgs &a, unsigned long long *sums, double *partial, hipStream_t s);
void launch_centroid_center(const VoroArgs &a, double *partial, hipStream_t s);
// cell normals and the partial sums of the enclosed volume (volume_partials of them), whose address is returned
const double *launch_volume_cells(const VoroArgs &a, unsigned long long *sums, double *normals, double *partial,
                                  hipStream_t s);
long long volume_partials(long long ncell);
// scal: [0] V, [1] push = strength (target - V) / target
void launch_volume_force(const VoroArgs &a, const double *vol_partial, double *scal, double target, double strength,
                         hipStream_t s);
void launch_volume_push(const VoroArgs &a, const double *normals, const double *fpush, double *f64, float *f32,
                        hipStream_t s);

}  // namespace orbc

#define ORBC_HIP_CHECK(expr)                                                     \
    do {                                                                         \
        hipError_t e_ = (expr);                                                  \
        if (e_ != hipSuccess) throw orbc::HipError(e_, #expr, __FILE__, __LINE__); \
    } while (0)

namespace orbc {
struct HipError {
    hipError_t err;
    const char *expr, *file;
    int line;
    HipError(hipError_t e, const char *x, const char *f, int l) : err(e), expr(x), file(f), line(l) {}
};
}  // namespace orbc
