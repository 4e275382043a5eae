// k_force.hip -- pair and bond forces, and the fused timestep kernel, gfx950.
//
// One lane owns one particle i (the reference's owner-computes rule across
// thread chunks, src/compute_pairwise_fused.h:249-316, applied to every
// pair): it walks its full neighbour list (tiled by particle block, list_base, so
// that the k-th entries of a wavefront's 64 particles are one coalesced
// 256-byte load),
// accumulates f_i and the director force t_i in registers and writes them
// once.  No atomics, fixed summation order: results are deterministic.
//
// Pair terms (src/pairwise_kernel.h:30-68, src/pairwise_kernel_fused.h:22-97):
//   anisotropic 4-8 polynomial when a lipid is involved, isotropic repulsive
//   polynomial between proteins, else WCA Lennard-Jones; selection
//   1e-5 < r^2 < rc^2 with the polynomial tested first
//   (src/compute_pairwise_fused.h:210,273-276,302-305).
// Bonds (src/compute_bonded.h:108-135): F_i = K (1 - r0/r) (x_j - x_i), each
//   end accumulated by its owner from a per-particle bond list.
//
// Precision: MIXED reads FP32 mirrors, whose positions are offsets from an
// integer anchor grid: selection, bonds and the rare isotropic terms in FP32, the
// anisotropic term in FP64 on the mirrors' exact separation.  FP64 evaluates
// everything in FP64 from the state itself.  The integrator update and all reductions are FP64 in both.
#include <type_traits>

#include "orbc_internal.h"

namespace orbc {

void upload_mass(const double *mass, hipStream_t s);   // k_integrate.hip

namespace {

__constant__ FFTab<float> c_fff;
__constant__ FFTab<double> c_ffd;

template <typename R> __device__ inline const FFTab<R> &ff();
template <> __device__ inline const FFTab<float> &ff<float>() { return c_fff; }
template <> __device__ inline const FFTab<double> &ff<double>() { return c_ffd; }

struct Acc {
    double fx = 0, fy = 0, fz = 0, tx = 0, ty = 0, tz = 0, e = 0, w = 0;
    double s = 0;              // FP64: force along the owner's director (pair_term), added by finish()
};

__device__ inline float rsq(float x) { return __builtin_amdgcn_rsqf(x); }

// exact-rounding helpers: the exported selection test must round exactly as the oracle
__device__ inline float sub_rn(float a, float b) { return __fsub_rn(a, b); }
__device__ inline double sub_rn(double a, double b) { return __dsub_rn(a, b); }
__device__ inline double add_rn(double a, double b) { return __dadd_rn(a, b); }
__device__ inline float r2_rn(float x, float y, float z) { return __fmaf_rn(z, z, __fmaf_rn(y, y, __fmul_rn(x, x))); }
__device__ inline double r2_rn(double x, double y, double z) { return __fma_rn(z, z, __fma_rn(y, y, __dmul_rn(x, x))); }

// |d| from r2 = |d|^2: rinv by the hardware reciprocal square root, then one
// Newton step on r so that r - r0 of a bond carries the rounding of r2 only.
__device__ inline void radius(float r2, float &r, float &rinv) {
    rinv = rsq(r2);
    r = r2 * rinv;
    r = __fmaf_rn(0.5f * __fmaf_rn(-r, r, r2), rinv, r);
}
__device__ inline void radius(double r2, double &r, double &rinv) {
    rinv = rsqrt(r2);
    r = r2 * rinv;
}

// ---- mixed pair terms ----------------------------------------------------------
// The radial factor carries (cut - r)^7 and A = 1 + alpha (a - 1) with alpha up
// to 5, so FP32 rounding of r, cut or a is amplified into relative errors near
// 1e-6 on the stiff lipid-protein terms.  The anisotropic term is therefore
// evaluated and summed in FP64 from the exact separation of the FP32 mirrors
// (X = (r_i - r_j) + h dA, formed in FP64 without rounding) and the FP32
// directors; FP64 and FP32 multiply-adds issue at the same rate here.  The
// selection test is FP32, as the oracle has it bit for bit.
//
// Everything one type pair needs, in three 16-byte LDS words.  alpha > 0 marks an
// anisotropic pair; the FP32 values of the other pairs (the FP64 ones rounded, as
// in the FP32 tables) lie two to a word.
typedef double Word2 __attribute__((ext_vector_type(2)));
struct PairRec {
    Word2 sel;         // alpha; (squared cutoffs of the polynomial, of the WCA)
    Word2 a;           // cut, 8 rep; or (cut, rep), (lj1, lj2)
    Word2 b;           // att, 4 att
};
static_assert(sizeof(PairRec) == 48, "three 16-byte LDS words");

__device__ inline double pack2(float lo, float hi) { return __hiloint2double(__float_as_int(hi), __float_as_int(lo)); }
__device__ inline float2 unpack2(double w) {
    return make_float2(__int_as_float(__double2loint(w)), __int_as_float(__double2hiint(w)));
}

__device__ inline void load_pair_recs(PairRec *s) {
    for (int k = threadIdx.x; k < NT * NT; k += blockDim.x) {
        const bool aniso = c_ffd.cut2_poly[k] > 0.0 && c_ffd.aniso[k];
        PairRec r;
        r.sel = Word2{aniso ? (double)c_fff.alpha[k] : 0.0, pack2(c_fff.cut2_poly[k], c_fff.cut2_lj[k])};
        r.a = aniso ? Word2{c_ffd.cut_poly[k], 8.0 * c_ffd.rep[k]}
                    : Word2{pack2((float)c_ffd.cut_poly[k], (float)c_ffd.rep[k]), pack2(c_fff.lj1[k], c_fff.lj2[k])};
        r.b = Word2{c_ffd.att[k], 4.0 * c_ffd.att[k]};
        s[k] = r;
    }
}

// Anisotropic polynomial term of one directed pair inside its cutoff
// (src/pairwise_kernel.h:37-62): force on i, director force on i, energy and
// virial halves; r2 the FP32 squared distance of the selection test
template <bool ENERGY>
__device__ __forceinline__ void aniso_fp64(const PairRec &P, float r2, double X, double Y, double Z,
                                           const double (&ni)[3], float njx, float njy, float njz, Acc &acc) {
    const double cut = P.a.x, rep8 = P.a.y, att = P.b.x, att4 = P.b.y, alpha = P.sel.x;
    const double d2 = __fma_rn(Z, Z, __fma_rn(Y, Y, X * X));
    double y = (double)rsq(r2);                               // 1/r to FP32 accuracy
    y = y * __fma_rn(-0.5 * d2, y * y, 1.5);                  // one Newton step: FP64 accuracy
    const double rd = d2 * y;
    const double ex = X * y, ey = Y * y, ez = Z * y;
    const double ax = ni[0], ay = ni[1], az = ni[2], bx = njx, by = njy, bz = njz;
    const double ninj = __fma_rn(az, bz, __fma_rn(ay, by, ax * bx));
    const double nie = __fma_rn(az, ez, __fma_rn(ay, ey, ax * ex));
    const double nje = __fma_rn(bz, ez, __fma_rn(by, ey, bx * ex));
    const double a = __fma_rn(-nie, nje, ninj);
    const double pix = __fma_rn(-nie, ex, ax), piy = __fma_rn(-nie, ey, ay), piz = __fma_rn(-nie, ez, az);
    const double pjx = __fma_rn(-nje, ex, bx), pjy = __fma_rn(-nje, ey, by), pjz = __fma_rn(-nje, ez, bz);
    const double s = cut - rd;
    const double s2 = s * s, s3 = s2 * s, s4 = s2 * s2;
    const double A = __fma_rn(alpha, a - 1.0, 1.0);
    const double aua = alpha * (att * s4);
    const double auar = aua * y;
    const double fra = s3 * __fma_rn(A, att4, rep8 * s4);
    const double fx = __fma_rn(fra, ex, auar * __fma_rn(nje, pix, nie * pjx));
    const double fy = __fma_rn(fra, ey, auar * __fma_rn(nje, piy, nie * pjy));
    const double fz = __fma_rn(fra, ez, auar * __fma_rn(nje, piz, nie * pjz));
    acc.tx -= (aua * pjx);
    acc.ty -= (aua * pjy);
    acc.tz -= (aua * pjz);
    acc.fx += fx; acc.fy += fy; acc.fz += fz;
    if (ENERGY) {
        acc.e += (0.5 * s4 * __fma_rn(A, att, 0.125 * rep8 * s4));
        acc.w += (0.5 * __fma_rn(Z, fz, __fma_rn(Y, fy, X * fx)));
    }
}

// Repulsive protein-protein polynomial, src/pairwise_kernel_fused.h:79-97, and
// WCA Lennard-Jones, :63-77, in FP32
template <bool ENERGY>
__device__ __forceinline__ void pp_term(float cutp, float rep, float r2, float dx, float dy, float dz,
                                        float &fx, float &fy, float &fz, Acc &acc) {
    float r, rinv;
    radius(r2, r, rinv);
    const float ex = dx * rinv, ey = dy * rinv, ez = dz * rinv;
    const float s = cutp - r;
    const float s3 = s * s * s, s4 = (s * s) * (s * s);
    const float fr = 8.0f * rep * s3 * s4;
    fx = fr * ex; fy = fr * ey; fz = fr * ez;
    if (ENERGY) acc.e += (double)(0.5f * rep * s4 * s4);
}

template <bool ENERGY>
__device__ __forceinline__ void lj_term(float lj1, float lj2, float r2, float dx, float dy, float dz, float &fx,
                                        float &fy, float &fz, Acc &acc) {
    const float r2inv = 1.0f / r2;
    const float r6inv = r2inv * r2inv * r2inv;
    const float fpair = r6inv * (lj1 * r6inv - lj2) * r2inv;
    fx = dx * fpair; fy = dy * fpair; fz = dz * fpair;
    if (ENERGY) acc.e += (double)(0.5f * r6inv * (lj1 * (1.0f / 12.0f) * r6inv - lj2 * (1.0f / 6.0f)));
}

// One directed pair (owner i, neighbour j) from the mirrors; ni: the owner's
// director in FP64.  The kind of pair is the first thing to branch on: the sums
// are then updated in place (after a branch on the distance they are copied
// first) and the record's words are read together instead of one after another
// test.  With the row read without branches (range_halo), 3.2 M particles 431 ->
// 408 us a launch, Nose-Hoover on 1.3 M 156 -> 132, one block alone 16.4 -> 12.7
// (averages with the launches that find the list spent, a seventh to a fifth of all).
template <bool ENERGY>
__device__ __forceinline__ void pair_rec(const Anchor &ag, const AnchorI &ai, float4 xi, const double (&ni)[3],
                                         float4 xj, float4 nj, const PairRec &P, Acc &acc) {
    const AnchorI aj = anchor_unpack(__float_as_uint(xj.w), ag);
    const float dx = anchor_add(ag, 0, sub_rn(xi.x, xj.x), ai.x - aj.x);
    const float dy = anchor_add(ag, 1, sub_rn(xi.y, xj.y), ai.y - aj.y);
    const float dz = anchor_add(ag, 2, sub_rn(xi.z, xj.z), ai.z - aj.z);
    const float r2 = r2_rn(dx, dy, dz);
    const float2 cut2 = unpack2(P.sel.y);
    if (P.sel.x > 0.0) {
        if (r2 > 1e-5f && r2 < cut2.x) {
            const double X = anchor_add_exact(ag, 0, xi.x, xj.x, ai.x - aj.x);
            const double Y = anchor_add_exact(ag, 1, xi.y, xj.y, ai.y - aj.y);
            const double Z = anchor_add_exact(ag, 2, xi.z, xj.z, ai.z - aj.z);
            aniso_fp64<ENERGY>(P, r2, X, Y, Z, ni, nj.x, nj.y, nj.z, acc);
        }
        return;
    }
    if (!(r2 > 1e-5f)) return;
    float fx, fy, fz;
    if (r2 < cut2.x) {
        const float2 c = unpack2(P.a.x);
        pp_term<ENERGY>(c.x, c.y, r2, dx, dy, dz, fx, fy, fz, acc);
    } else {
        if (!(r2 < cut2.y)) return;
        const float2 lj = unpack2(P.a.y);
        lj_term<ENERGY>(lj.x, lj.y, r2, dx, dy, dz, fx, fy, fz, acc);
    }
    acc.fx = add_rn(acc.fx, (double)fx); acc.fy = add_rn(acc.fy, (double)fy); acc.fz = add_rn(acc.fz, (double)fz);
    if (ENERGY) acc.w += (double)(0.5f * __fmaf_rn(dz, fz, __fmaf_rn(dy, fy, __fmul_rn(dx, fx))));
}

// ---- FP64 pair terms -------------------------------------------------------------
// 1 / sqrt(d2): the FP32 hardware estimate and one third-order step (relative
// error of the estimate 1.2e-7, its cube is far below FP64 rounding).  d2 lies
// within a few cutoffs squared of 1, far from the ends of the FP32 range.
__device__ __forceinline__ double inv_sqrt(double d2) {
#pragma clang fp contract(off)
    const double y = (double)rsq((float)d2);
    const double h = __builtin_fma(-d2 * y, y, 1.0);
    return __builtin_fma(y * h, __builtin_fma(0.375, h, 0.5), y);
}

// Constants of one type pair, three 16-byte LDS words read together.  A pair
// type interacts by one term only: the anisotropic polynomial (alpha > 0), the
// repulsive polynomial between proteins (cut > 0) or WCA Lennard-Jones.
struct PairRec64 {
    Word2 sel;                 // squared cutoff of the term; alpha
    Word2 a;                   // polynomial cutoff (0: Lennard-Jones); alpha att, or lj1
    Word2 b;                   // 4 att, or lj2; 8 rep
};
static_assert(sizeof(PairRec64) == 48, "three 16-byte LDS words");

__device__ inline void load_pair_recs(PairRec64 *s) {
    for (int k = threadIdx.x; k < NT * NT; k += blockDim.x) {
        PairRec64 r;
        const bool poly = c_ffd.cut2_poly[k] > 0.0, aniso = poly && c_ffd.aniso[k];
        r.sel = Word2{poly ? c_ffd.cut2_poly[k] : c_ffd.cut2_lj[k], aniso ? c_ffd.alpha[k] : 0.0};
        r.a = Word2{poly ? c_ffd.cut_poly[k] : 0.0, aniso ? c_ffd.alpha[k] * c_ffd.att[k] : c_ffd.lj1[k]};
        r.b = Word2{aniso ? 4.0 * c_ffd.att[k] : c_ffd.lj2[k], 8.0 * c_ffd.rep[k]};
        s[k] = r;
    }
}

// One directed pair, owner i and neighbour j, from X = x_i - x_j; nothing
// unless 1e-5 < |X|^2 < rc^2.  Every multiply-add is written out (and the
// compiler forms none of its own), so the walks below -- 32-bit or 16-bit list,
// gathered or staged -- give the same bits.
//
// Anisotropic term (src/pairwise_kernel.h:37-62): with e = X / r, a = n_i.n_j -
// (n_i.e)(n_j.e), s = cut - r and u = alpha att s^4,
//   f = c_e e + u/r ((n_j.e) n_i + (n_i.e) n_j),
//   t = -u (n_j - (n_j.e) e),
// where c_e gathers the radial force and the e parts of the projections p_i,
// p_j that the reference forms as vectors.  The n_i part of f is summed as the
// scalar s and applied once per particle (finish): 50 operations a pair from the
// separation on, a multiply-add counted once, against 57 with the vectors p_i,
// p_j, e and f formed (aniso_fp64).
__device__ __forceinline__ void pair_term(const PairRec64 &P, double X, double Y, double Z, const double (&ni)[3],
                                          double bx, double by, double bz, Acc &acc) {
#pragma clang fp contract(off)
    const double d2 = __builtin_fma(Z, Z, __builtin_fma(Y, Y, X * X));
    if (!(d2 < P.sel.x && d2 > 1e-5)) return;
    if (P.sel.y > 0.0) {
        const double y = inv_sqrt(d2), r = d2 * y;
        const double ninj = __builtin_fma(ni[2], bz, __builtin_fma(ni[1], by, ni[0] * bx));
        const double nie = __builtin_fma(ni[2], Z, __builtin_fma(ni[1], Y, ni[0] * X)) * y;
        const double nje = __builtin_fma(bz, Z, __builtin_fma(by, Y, bx * X)) * y;
        const double A = __builtin_fma(P.sel.y, __builtin_fma(-nie, nje, ninj) - 1.0, 1.0);
        const double s = P.a.x - r, s2 = s * s, s4 = s2 * s2, s3 = s2 * s;
        const double u = P.a.y * s4, uy = u * y;
        const double fra = s3 * __builtin_fma(A, P.b.x, P.b.y * s4);
        const double ci = uy * nje, cj = uy * nie;
        const double cx = __builtin_fma(-2.0 * ci, nie, fra) * y;
        acc.fx = __builtin_fma(cx, X, __builtin_fma(cj, bx, acc.fx));
        acc.fy = __builtin_fma(cx, Y, __builtin_fma(cj, by, acc.fy));
        acc.fz = __builtin_fma(cx, Z, __builtin_fma(cj, bz, acc.fz));
        acc.s += ci;
        acc.tx = __builtin_fma(ci, X, __builtin_fma(-u, bx, acc.tx));
        acc.ty = __builtin_fma(ci, Y, __builtin_fma(-u, by, acc.ty));
        acc.tz = __builtin_fma(ci, Z, __builtin_fma(-u, bz, acc.tz));
        return;
    }
    double c;                  // f = c X
    if (P.a.x > 0.0) {
        // src/pairwise_kernel_fused.h:79-97
        const double y = inv_sqrt(d2), s = P.a.x - d2 * y, s2 = s * s, s4 = s2 * s2;
        c = P.b.y * (s4 * (s2 * s)) * y;
    } else {
        // src/pairwise_kernel_fused.h:63-77
        const double q = 1.0 / d2, q3 = q * q * q;
        c = q3 * __builtin_fma(P.a.y, q3, -P.b.x) * q;
    }
    acc.fx = __builtin_fma(c, X, acc.fx);
    acc.fy = __builtin_fma(c, Y, acc.fy);
    acc.fz = __builtin_fma(c, Z, acc.fz);
}

// after a particle's last pair
__device__ __forceinline__ void finish(const double (&ni)[3], Acc &acc) {
#pragma clang fp contract(off)
    acc.fx = __builtin_fma(acc.s, ni[0], acc.fx);
    acc.fy = __builtin_fma(acc.s, ni[1], acc.fy);
    acc.fz = __builtin_fma(acc.s, ni[2], acc.fz);
}

// minimum image on the periodic axes
__device__ __forceinline__ void image(const Anchor &a, double &X, double &Y, double &Z) {
#pragma clang fp contract(off)
    if (a.L[0] > 0) X = __builtin_fma(-a.L[0], rint(X * a.Linv[0]), X);
    if (a.L[1] > 0) Y = __builtin_fma(-a.L[1], rint(Y * a.Linv[1]), Y);
    if (a.L[2] > 0) Z = __builtin_fma(-a.L[2], rint(Z * a.Linv[2]), Z);
}
__device__ inline bool is_periodic(const Anchor &a) { return a.L[0] > 0 || a.L[1] > 0 || a.L[2] > 0; }

// bond constants in LDS
template <typename R>
struct BondTab {
    R K[NBT], r0[NBT];
};
template <typename R>
__device__ inline void load_bonds(BondTab<R> &t) {
    if (threadIdx.x < NBT) { t.K[threadIdx.x] = ff<R>().bond_K[threadIdx.x]; t.r0[threadIdx.x] = ff<R>().bond_r0[threadIdx.x]; }
}

template <typename R>
struct BondAcc {
    R fx = 0, fy = 0, fz = 0, e = 0, w = 0;
};
template <typename R>
__device__ inline void add_to(Acc &o, const BondAcc<R> &a) {
    o.fx += (double)a.fx; o.fy += (double)a.fy; o.fz += (double)a.fz;
    o.e += (double)a.e; o.w += (double)a.w;
}
template <typename R, bool ENERGY, typename TAB>
__device__ __forceinline__ void bond_ij(const TAB &t, int bt, R dx, R dy, R dz, BondAcc<R> &acc) {
    const R r2 = dx * dx + dy * dy + dz * dz;
    R r, rinv;
    radius(r2, r, rinv);
    const R K = t.K[bt], r0 = t.r0[bt];
    const R c = K * ((r - r0) * rinv);
    acc.fx += c * dx; acc.fy += c * dy; acc.fz += c * dz;
    if (ENERGY) {
        const R dr = r - r0;
        acc.e += R(0.25) * K * dr * dr;
        acc.w += R(-0.5) * c * r2;
    }
}

__device__ inline long long block_index(int swizzle) {
    const unsigned b = blockIdx.x, nb = gridDim.x;
    if (!swizzle) return b;
    // consecutive particle tiles on one XCD (blocks are dealt round-robin over
    // the 8 XCDs), so neighbour gathers hit that XCD's L2
    const unsigned q = nb >> 3, r = nb & 7u, xcd = b & 7u, k = b >> 3;
    return (xcd < r) ? (long long)xcd * (q + 1) + k : (long long)r * (q + 1) + (long long)(xcd - r) * q + k;
}

__device__ inline AnchorI unpack(uint32_t w, const Anchor &a) { return anchor_unpack(w, a); }

// Neighbours gathered per group in the walks over the 32-bit list (loads in
// flight per wave: mixed 3, with the next group gathered while this one is
// evaluated, 0.574 ms against 0.594 for 2 and 0.613 for 4 unpipelined on the
// full RBC).
constexpr int UNROLL_MIXED = 3;
constexpr int UNROLL64 = 4;

// ---- per-particle force accumulation ---------------------------------------
// The list is walked in groups of that many entries; a group is padded with the
// particle itself (distance 0, no contribution).

// pairs of particle i over the 32-bit list, mixed
template <bool ENERGY, int UNROLL = UNROLL_MIXED>
__device__ __forceinline__ void pairs_mixed(long long i, int kmax, const PQ *pq, const uint32_t *nbr,
                                            const uint32_t *nnbr, const Anchor &ag, const PairRec *recs, Acc &acc) {
    const PQ qi = pq[i];
    const AnchorI ai = unpack(__float_as_uint(qi.x.w), ag);
    const PairRec *const row = recs + __float_as_int(qi.n.w) * NT;
    const double ni[3] = {qi.n.x, qi.n.y, qi.n.z};
    const int nr = (int)nnbr[i];
    const uint32_t *const nb = nbr + list_base(i, kmax);
    if constexpr (UNROLL == 1) {
        for (int k = 0; k < nr; ++k) {
            const PQ q = pq[nb[k * BLOCK]];
            pair_rec<ENERGY>(ag, ai, qi.x, ni, q.x, q.n, row[__float_as_int(q.n.w)], acc);
        }
        return;
    }
    uint32_t jn[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) jn[u] = u < nr ? nb[u * BLOCK] : (uint32_t)i;
    float4 xa[UNROLL], na[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) { xa[u] = pq[jn[u]].x; na[u] = pq[jn[u]].n; }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) jn[u] = UNROLL + u < nr ? nb[(UNROLL + u) * BLOCK] : (uint32_t)i;
    for (int k0 = 0; k0 < nr; k0 += UNROLL) {
        float4 xb[UNROLL], nbv[UNROLL];
        const bool more = k0 + UNROLL < nr;
        if (more) {
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) { xb[u] = pq[jn[u]].x; nbv[u] = pq[jn[u]].n; }
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) {
                const int kn = k0 + 2 * UNROLL + u;
                jn[u] = kn < nr ? nb[kn * BLOCK] : (uint32_t)i;
            }
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
            pair_rec<ENERGY>(ag, ai, qi.x, ni, xa[u], na[u], row[__float_as_int(na[u].w)], acc);
        if (more) {
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) { xa[u] = xb[u]; na[u] = nbv[u]; }
        }
    }
}

// the same in FP64
__device__ __forceinline__ void pairs_fp64(long long i, int kmax, const double *x, const double *nrm,
                                           const uint8_t *type, const uint32_t *nbr, const uint32_t *nnbr,
                                           const Anchor &ag, const PairRec64 *recs, Acc &acc) {
    const double xi = x[3 * i], yi = x[3 * i + 1], zi = x[3 * i + 2];
    const double ni[3] = {nrm[3 * i], nrm[3 * i + 1], nrm[3 * i + 2]};
    const PairRec64 *const row = recs + type[i] * NT;
    const bool periodic = is_periodic(ag);
    const int nr = (int)nnbr[i];
    const uint32_t *const nb = nbr + list_base(i, kmax);
    long long jn[UNROLL64];
#pragma unroll
    for (int u = 0; u < UNROLL64; ++u) jn[u] = u < nr ? (long long)nb[u * BLOCK] : i;
    for (int k0 = 0; k0 < nr; k0 += UNROLL64) {
        double xj[UNROLL64][3], nj[UNROLL64][3];
        int tj[UNROLL64];
#pragma unroll
        for (int u = 0; u < UNROLL64; ++u) {
            const long long j = jn[u];
            for (int d = 0; d < 3; ++d) { xj[u][d] = x[3 * j + d]; nj[u][d] = nrm[3 * j + d]; }
            tj[u] = type[j];
            const int kn = k0 + UNROLL64 + u;
            jn[u] = kn < nr ? (long long)nb[kn * BLOCK] : i;
        }
#pragma unroll
        for (int u = 0; u < UNROLL64; ++u) {
            double X = xi - xj[u][0], Y = yi - xj[u][1], Z = zi - xj[u][2];
            if (periodic) image(ag, X, Y, Z);
            pair_term(row[tj[u]], X, Y, Z, ni, nj[u][0], nj[u][1], nj[u][2], acc);
        }
    }
    finish(ni, acc);
}

// Bonds of a particle, four at a time: their entries, then their partners'
// positions, are loaded together (one after the other each bond waits for two
// loads), the terms are summed in list order.
constexpr int BOND_GROUP = 4;

// compute_bonded from the FP32 mirrors (f only); TAB holds K[] and r0[]
template <bool ENERGY, typename TAB>
__device__ __forceinline__ void bonds_mixed(long long i, int nb, long long stride, const PQ *pq, const uint32_t *bnd,
                                            const Anchor &ag, const TAB &t, Acc &out) {
    if (nb == 0) return;
    const float4 xi = pq[i].x;
    const AnchorI ai = unpack(__float_as_uint(xi.w), ag);
    BondAcc<float> acc;
    for (int k0 = 0; k0 < nb; k0 += BOND_GROUP) {
        uint32_t e[BOND_GROUP];
        float4 xj[BOND_GROUP];
#pragma unroll
        for (int u = 0; u < BOND_GROUP; ++u) e[u] = k0 + u < nb ? bnd[(long long)(k0 + u) * stride + i] : (uint32_t)i;
#pragma unroll
        for (int u = 0; u < BOND_GROUP; ++u) xj[u] = pq[e[u] & BOND_INDEX_MASK].x;
#pragma unroll
        for (int u = 0; u < BOND_GROUP; ++u) {
            if (k0 + u >= nb) break;
            const AnchorI aj = unpack(__float_as_uint(xj[u].w), ag);
            const float dx = anchor_add(ag, 0, sub_rn(xj[u].x, xi.x), aj.x - ai.x);
            const float dy = anchor_add(ag, 1, sub_rn(xj[u].y, xi.y), aj.y - ai.y);
            const float dz = anchor_add(ag, 2, sub_rn(xj[u].z, xi.z), aj.z - ai.z);
            bond_ij<float, ENERGY>(t, (int)(e[u] >> 30), dx, dy, dz, acc);
        }
    }
    add_to(out, acc);
}

// compute_bonded in FP64
template <typename TAB>
__device__ __forceinline__ void bonds_fp64(long long i, int nb, long long stride, const double *x, const uint32_t *bnd,
                                           const Anchor &ag, const TAB &t, Acc &out) {
    if (nb == 0) return;
    const double xi = x[3 * i], yi = x[3 * i + 1], zi = x[3 * i + 2];
    BondAcc<double> acc;
    for (int k0 = 0; k0 < nb; k0 += BOND_GROUP) {
        uint32_t e[BOND_GROUP];
        double xj[BOND_GROUP][3];
#pragma unroll
        for (int u = 0; u < BOND_GROUP; ++u) e[u] = k0 + u < nb ? bnd[(long long)(k0 + u) * stride + i] : (uint32_t)i;
#pragma unroll
        for (int u = 0; u < BOND_GROUP; ++u) {
            const long long j = e[u] & BOND_INDEX_MASK;
            for (int d = 0; d < 3; ++d) xj[u][d] = x[3 * j + d];
        }
#pragma unroll
        for (int u = 0; u < BOND_GROUP; ++u) {
            if (k0 + u >= nb) break;
            double dx = xj[u][0] - xi, dy = xj[u][1] - yi, dz = xj[u][2] - zi;
            image(ag, dx, dy, dz);
            bond_ij<double, false>(t, (int)(e[u] >> 30), dx, dy, dz, acc);
        }
    }
    add_to(out, acc);
}

// ---- FP64 forces of the per-call entry points ---------------------------------
// Apart from pair_term and in plain expressions: the minimiser descends along
// these forces, and within some 300 of its capped steps a difference in the
// last bit grows to 1e-3 of the positions, so a relaxed start is reproduced
// only by the same operations in the same order.
namespace plain {
struct Acc {
    double fx = 0, fy = 0, fz = 0, tx = 0, ty = 0, tz = 0, e = 0, w = 0;
};
struct Tab {
    double cut2p[36], cutp[36], rep[36], att[36], alpha[36], cut2lj[36], lj1[36], lj2[36];
    int aniso[36];
    double K[NBT], r0[NBT];
};

__device__ inline void load_tab(Tab *s) {
    const FFTab<double> &t = c_ffd;
    for (int k = threadIdx.x; k < 36; k += blockDim.x) {
        s->cut2p[k] = t.cut2_poly[k]; s->cutp[k] = t.cut_poly[k]; s->rep[k] = t.rep[k]; s->att[k] = t.att[k];
        s->alpha[k] = t.alpha[k]; s->cut2lj[k] = t.cut2_lj[k]; s->lj1[k] = t.lj1[k]; s->lj2[k] = t.lj2[k];
        s->aniso[k] = t.aniso[k];
    }
    if (threadIdx.x < NBT) { s->K[threadIdx.x] = t.bond_K[threadIdx.x]; s->r0[threadIdx.x] = t.bond_r0[threadIdx.x]; }
    __syncthreads();
}

// src/pairwise_kernel.h:37-62
template <bool ENERGY>
__device__ __forceinline__ void aniso_plain(const Tab &t, int k, double r2, double dx, double dy, double dz,
                                            double nix, double niy, double niz, double njx, double njy, double njz,
                                            Acc &acc) {
    double r, rinv;
    radius(r2, r, rinv);
    const double alpha = t.alpha[k];
    const double ex = dx * rinv, ey = dy * rinv, ez = dz * rinv;
    const double ninj = nix * njx + niy * njy + niz * njz;
    const double nie = nix * ex + niy * ey + niz * ez;
    const double nje = njx * ex + njy * ey + njz * ez;
    const double a = ninj - nie * nje;
    const double pix = nix - nie * ex, piy = niy - nie * ey, piz = niz - nie * ez;
    const double pjx = njx - nje * ex, pjy = njy - nje * ey, pjz = njz - nje * ez;
    double fra, aua, auar, en = 0.0;
    const double s = t.cutp[k] - r;
    const double s2 = s * s, s3 = s2 * s, s4 = s2 * s2;
    const double A = 1.0 + alpha * (a - 1.0);
    const double rep = t.rep[k], att = t.att[k];
    aua = alpha * (att * s4);
    auar = aua * rinv;
    fra = s3 * (8.0 * rep * s4 + 4.0 * A * att);
    if (ENERGY) en = 0.5 * s4 * (rep * s4 + A * att);
    const double fx = fra * ex + auar * (nje * pix + nie * pjx);
    const double fy = fra * ey + auar * (nje * piy + nie * pjy);
    const double fz = fra * ez + auar * (nje * piz + nie * pjz);
    acc.tx -= (aua * pjx);
    acc.ty -= (aua * pjy);
    acc.tz -= (aua * pjz);
    acc.fx += fx; acc.fy += fy; acc.fz += fz;
    if (ENERGY) {
        acc.e += en;
        acc.w += (0.5 * (dx * fx + dy * fy + dz * fz));
    }
}

template <bool ENERGY>
__device__ __forceinline__ void pair_plain(const Tab &t, int ti, int tj, double dx, double dy, double dz, double r2,
                                           double nix, double niy, double niz, double njx, double njy, double njz,
                                           Acc &acc) {
    if (!(r2 > 1e-5)) return;
    const int k = ti * NT + tj;
    double fx, fy, fz;
    if (r2 < t.cut2p[k]) {
        if (t.aniso[k]) {
            aniso_plain<ENERGY>(t, k, r2, dx, dy, dz, nix, niy, niz, njx, njy, njz, acc);
            return;
        }
        // src/pairwise_kernel_fused.h:79-97
        double r, rinv;
        radius(r2, r, rinv);
        const double ex = dx * rinv, ey = dy * rinv, ez = dz * rinv;
        const double s = t.cutp[k] - r;
        const double s3 = s * s * s, s4 = (s * s) * (s * s);
        const double rep = t.rep[k];
        const double fr = 8.0 * rep * s3 * s4;
        fx = fr * ex; fy = fr * ey; fz = fr * ez;
        if (ENERGY) acc.e += (0.5 * rep * s4 * s4);
    } else {
        if (!(r2 < t.cut2lj[k])) return;
        // src/pairwise_kernel_fused.h:63-77
        const double r2inv = 1.0 / r2;
        const double r6inv = r2inv * r2inv * r2inv;
        const double fpair = r6inv * (t.lj1[k] * r6inv - t.lj2[k]) * r2inv;
        fx = dx * fpair; fy = dy * fpair; fz = dz * fpair;
        if (ENERGY) acc.e += (0.5 * r6inv * (t.lj1[k] * (1.0 / 12.0) * r6inv - t.lj2[k] * (1.0 / 6.0)));
    }
    acc.fx += fx; acc.fy += fy; acc.fz += fz;
    if (ENERGY) acc.w += (0.5 * (dx * fx + dy * fy + dz * fz));
}

template <bool ENERGY>
__device__ __forceinline__ void bond_plain(const Tab &t, int bt, double dx, double dy, double dz, Acc &acc) {
    const double r2 = dx * dx + dy * dy + dz * dz;
    double r, rinv;
    radius(r2, r, rinv);
    const double K = t.K[bt], r0 = t.r0[bt];
    const double c = K * ((r - r0) * rinv);
    acc.fx += c * dx; acc.fy += c * dy; acc.fz += c * dz;
    if (ENERGY) {
        const double dr = r - r0;
        acc.e += 0.25 * K * dr * dr;
        acc.w += -0.5 * c * r2;
    }
}

template <bool ENERGY>
__device__ __forceinline__ void accumulate(long long i, long long stride, int kmax, const double *x, const double *nrm,
                                           const uint8_t *type, const uint32_t *nbr, const uint32_t *nnbr,
                                           const uint32_t *bnd, const uint8_t *nbnd, const Anchor &ag, const Tab &t,
                                           Acc &acc, bool pair, bool bond) {
    const double xi = x[3 * i], yi = x[3 * i + 1], zi = x[3 * i + 2];
    if (pair) {
        const double nix = nrm[3 * i], niy = nrm[3 * i + 1], niz = nrm[3 * i + 2];
        const int ti = type[i], ke = (int)nnbr[i];
        const bool periodic = is_periodic(ag);
        const uint32_t *const nb = nbr + list_base(i, kmax);
        long long jn[UNROLL64];
#pragma unroll
        for (int u = 0; u < UNROLL64; ++u) jn[u] = u < ke ? (long long)nb[u * BLOCK] : i;
        for (int k0 = 0; k0 < ke; k0 += UNROLL64) {
            double xj[UNROLL64][3], nj[UNROLL64][3];
            int tj[UNROLL64];
#pragma unroll
            for (int u = 0; u < UNROLL64; ++u) {
                const long long j = jn[u];
                for (int d = 0; d < 3; ++d) { xj[u][d] = x[3 * j + d]; nj[u][d] = nrm[3 * j + d]; }
                tj[u] = type[j];
                const int kn = k0 + UNROLL64 + u;
                jn[u] = kn < ke ? (long long)nb[kn * BLOCK] : i;
            }
#pragma unroll
            for (int u = 0; u < UNROLL64; ++u) {
                double dx = sub_rn(xi, xj[u][0]);
                double dy = sub_rn(yi, xj[u][1]);
                double dz = sub_rn(zi, xj[u][2]);
                if (periodic) min_image(ag, dx, dy, dz);
                const double r2 = r2_rn(dx, dy, dz);
                pair_plain<ENERGY>(t, ti, tj[u], dx, dy, dz, r2, nix, niy, niz, nj[u][0], nj[u][1], nj[u][2], acc);
            }
        }
    }
    if (bond && nbnd) {
        const int nb = nbnd[i];
        for (int k = 0; k < nb; ++k) {
            const uint32_t e = bnd[(long long)k * stride + i];
            const long long j = e & BOND_INDEX_MASK;
            double dx = x[3 * j] - xi, dy = x[3 * j + 1] - yi, dz = x[3 * j + 2] - zi;
            min_image(ag, dx, dy, dz);
            bond_plain<ENERGY>(t, (int)(e >> 30), dx, dy, dz, acc);
        }
    }
}
}  // namespace plain

// ---- standalone force evaluation (compute_pairwise_fused / compute_bonded) --
template <bool MIXED, bool ENERGY>
__global__ __launch_bounds__(BLOCK) void k_forces(ForceArgs a, int pair, int bond) {
    if constexpr (MIXED) {
        __shared__ PairRec recs[NT * NT];
        __shared__ BondTab<float> bt;
        load_pair_recs(recs);
        load_bonds(bt);
        __syncthreads();
        const long long i = block_index(a.swizzle) * BLOCK + threadIdx.x;
        if (i >= a.n) return;
        Acc acc;
        if (pair) pairs_mixed<ENERGY>(i, a.kmax, a.pq, a.nbr, a.nnbr, a.anc_grid, recs, acc);
        if (bond && a.nbnd) bonds_mixed<ENERGY>(i, (int)a.nbnd[i], a.stride, a.pq, a.bnd, a.anc_grid, bt, acc);
        a.f32[3 * i] += (float)acc.fx; a.f32[3 * i + 1] += (float)acc.fy; a.f32[3 * i + 2] += (float)acc.fz;
        a.t32[3 * i] += (float)acc.tx; a.t32[3 * i + 1] += (float)acc.ty; a.t32[3 * i + 2] += (float)acc.tz;
        if (ENERGY) { a.e[i] += acc.e; a.w[i] += acc.w; }
    } else {
        __shared__ plain::Tab t;
        plain::load_tab(&t);
        const long long i = block_index(a.swizzle) * BLOCK + threadIdx.x;
        if (i >= a.n) return;
        plain::Acc acc;
        plain::accumulate<ENERGY>(i, a.stride, a.kmax, a.x, a.nrm, a.type, a.nbr, a.nnbr, a.bnd, a.nbnd, a.anc_grid, t,
                                  acc, pair, bond);
        a.f64[3 * i] += acc.fx; a.f64[3 * i + 1] += acc.fy; a.f64[3 * i + 2] += acc.fz;
        a.t64[3 * i] += acc.tx; a.t64[3 * i + 1] += acc.ty; a.t64[3 * i + 2] += acc.tz;
        if (ENERGY) { a.e[i] += acc.e; a.w[i] += acc.w; }
    }
}

// ---- one step of the minimiser -------------------------------------------------
// Forces and bonds as k_forces, then post_torque (src/integrate_nh.h:146-154), the
// capped steepest descent (src/openrbc.cpp:114-131) and bounce_back
// (src/integrate_nh.h:124-144) with the expressions of separate kernels, whose
// force arrays (FP32 in mixed precision) round f and n x t here too: the results
// are the same to the last bit.  Positions, directors and mirrors go to the other
// buffers, so a step needs no force arrays, no pass over the state for each stage
// and, with the skin check of k_disp and the step kernels' flags (StepArgs::dslot),
// no look at the list from the host: 20 steps of 227,000 particles in FP64 2.55 ->
// 1.67 ms, with four rebuilds whose block halos are now left out.  A step's 54 us
// wait for gathered neighbours.  Staged ones have not been tried here: the fused FP64
// step of these particles takes 52 us gathered and 34 staged, and building the
// halos 34, for lists that last some five steps.
// (The multiply-adds that the descent's last bits depend on are written out.)
__device__ inline void cross(const double *a, const double *b, double *c) {
    c[0] = __builtin_fma(a[1], b[2], -(a[2] * b[1]));
    c[1] = __builtin_fma(a[2], b[0], -(a[0] * b[2]));
    c[2] = __builtin_fma(a[0], b[1], -(a[1] * b[0]));
}
__device__ inline double norm(const double *a) {
    return sqrt(__builtin_fma(a[2], a[2], __builtin_fma(a[0], a[0], a[1] * a[1])));
}

template <bool MIXED>
__global__ __launch_bounds__(BLOCK) void k_min_step(MinArgs m) {
    const StepArgs &a = m.s;
    const Anchor &ag = a.anc_grid;
    const int k3 = (int)(a.step % 3ull);
    if (*a.stop || a.dslot[(k3 + 2) % 3] != 0u) {
        if (blockIdx.x == 0 && threadIdx.x == 0) *a.stop = 1;
        return;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        a.dslot[(k3 + 1) % 3] = 0u;
        atomicAdd(a.done, 1);
    }
    const long long i = block_index(a.swizzle) * BLOCK + threadIdx.x;
    double f[3], t[3];
    if constexpr (MIXED) {
        __shared__ PairRec recs[NT * NT];
        __shared__ BondTab<float> bt;
        load_pair_recs(recs);
        load_bonds(bt);
        __syncthreads();
        if (i < a.n) {
            Acc acc;
            pairs_mixed<false>(i, a.kmax, a.pq_in, a.nbr, a.nnbr, ag, recs, acc);
            if (a.nbnd) bonds_mixed<false>(i, (int)a.nbnd[i], a.stride, a.pq_in, a.bnd, ag, bt, acc);
            f[0] = (float)acc.fx; f[1] = (float)acc.fy; f[2] = (float)acc.fz;
            t[0] = (float)acc.tx; t[1] = (float)acc.ty; t[2] = (float)acc.tz;
        }
    } else {
        __shared__ plain::Tab tab;
        plain::load_tab(&tab);
        if (i < a.n) {
            plain::Acc acc;
            plain::accumulate<false>(i, a.stride, a.kmax, a.x_in, a.n_in, a.type, a.nbr, a.nnbr, a.bnd, a.nbnd, ag, tab,
                                     acc, true, a.has_bonds);
            f[0] = acc.fx; f[1] = acc.fy; f[2] = acc.fz;
            t[0] = acc.tx; t[1] = acc.ty; t[2] = acc.tz;
        }
    }
    bool past = false;
    if (i < a.n) {
        const int ty = a.type[i];
        const double mass = c_ffd.mass[ty];
        double x[3], n[3], q[3], dn[3];
        for (int d = 0; d < 3; ++d) { x[d] = a.x_in[3 * i + d]; n[d] = a.n_in[3 * i + d]; }
        const uint32_t w = a.anc[i];
        const float rb[3] = {a.rb[3 * i], a.rb[3 * i + 1], a.rb[3 * i + 2]};
        cross(n, t, q);
        if (MIXED)
            for (int d = 0; d < 3; ++d) q[d] = (float)q[d];
        cross(q, n, dn);
        const double ndx = norm(f) / mass, ndn = norm(dn);
        double h = a.dt;
        if (ndx > m.dr_opt || ndn > m.dn_opt) h = fmin(m.dr_opt / ndx, m.dn_opt / ndn);
        for (int d = 0; d < 3; ++d) { x[d] = __builtin_fma(f[d], h / mass, x[d]); n[d] = __builtin_fma(dn[d], h, n[d]); }
        const double s = 1.0 / norm(n);
        for (int d = 0; d < 3; ++d) n[d] *= s;
        for (int d = 0; d < 3; ++d) {
            if (ag.L[d] > 0) continue;              // periodic axis: no walls
            if (x[d] < m.box_lo[d]) { x[d] = m.box_lo[d] + (m.box_lo[d] - x[d]); a.v[3 * i + d] = -a.v[3 * i + d]; }
            else if (x[d] > m.box_hi[d]) { x[d] = m.box_hi[d] - (x[d] - m.box_hi[d]); a.v[3 * i + d] = -a.v[3 * i + d]; }
        }
        for (int d = 0; d < 3; ++d) { a.x_out[3 * i + d] = x[d]; a.n_out[3 * i + d] = n[d]; }
        const AnchorI A = unpack(w, ag);
        const float r[3] = {__double2float_rn(x[0] - anchor_pos(ag, 0, A.x)), __double2float_rn(x[1] - anchor_pos(ag, 1, A.y)),
                            __double2float_rn(x[2] - anchor_pos(ag, 2, A.z))};
        if (MIXED) {
            PQ p;
            p.x = make_float4(r[0], r[1], r[2], __uint_as_float(w));
            p.n = make_float4(__double2float_rn(n[0]), __double2float_rn(n[1]), __double2float_rn(n[2]), __int_as_float(ty));
            a.pq_out[i] = p;
        }
        float d2 = 0.f;
        for (int d = 0; d < 3; ++d) {
            const float e = r[d] - rb[d];
            d2 += e * e;
        }
        past = !((double)d2 <= m.half2);            // also when d2 is not a number
        if (past && isfinite(d2) && a.bud2 && a.nnbr[i] == 0 && a.bud2[i] > 0.f) past = d2 > a.bud2[i];
    }
    const unsigned long long over = __ballot(past);
    if (over && __lane_id() == (int)__ffsll((long long)over) - 1) atomicOr(a.dslot + k3, 1u);
}

template <bool MIXED>
__global__ __launch_bounds__(BLOCK) void k_pairs_export(ForceArgs a, unsigned *ids_i, unsigned *ids_j,
                                                        unsigned long long *count, long long cap) {
    const long long i = (long long)blockIdx.x * BLOCK + threadIdx.x;
    if (i >= a.n) return;
    const uint32_t idi = a.id[i];
    const int cnt = (int)a.nnbr[i];
    const uint32_t *const row = a.nbr + list_base(i, a.kmax);
    for (int k = 0; k < cnt; ++k) {
        const uint32_t j = row[k * BLOCK];
        const uint32_t idj = a.id[j];
        if (!(idi < idj)) continue;
        bool hit;
        if (MIXED) {
            const float4 xi = a.pq[i].x, xj = a.pq[j].x;
            const AnchorI ai = unpack(__float_as_uint(xi.w), a.anc_grid), aj = unpack(__float_as_uint(xj.w), a.anc_grid);
            const float dx = anchor_add(a.anc_grid, 0, sub_rn(xi.x, xj.x), ai.x - aj.x);
            const float dy = anchor_add(a.anc_grid, 1, sub_rn(xi.y, xj.y), ai.y - aj.y);
            const float dz = anchor_add(a.anc_grid, 2, sub_rn(xi.z, xj.z), ai.z - aj.z);
            const float r2 = r2_rn(dx, dy, dz);
            const int kk = __float_as_int(a.pq[i].n.w) * NT + __float_as_int(a.pq[j].n.w);
            hit = r2 > 1e-5f && (r2 < c_fff.cut2_poly[kk] || r2 < c_fff.cut2_lj[kk]);
        } else {
            double dx = sub_rn(a.x[3 * i], a.x[3 * (long long)j]);
            double dy = sub_rn(a.x[3 * i + 1], a.x[3 * (long long)j + 1]);
            double dz = sub_rn(a.x[3 * i + 2], a.x[3 * (long long)j + 2]);
            min_image(a.anc_grid, dx, dy, dz);
            const double r2 = r2_rn(dx, dy, dz);
            const int kk = a.type[i] * NT + a.type[j];
            hit = r2 > 1e-5 && (r2 < c_ffd.cut2_poly[kk] || r2 < c_ffd.cut2_lj[kk]);
        }
        if (hit) {
            const unsigned long long slot = atomicAdd(count, 1ull);
            if ((long long)slot < cap) { ids_i[slot] = idi; ids_j[slot] = idj; }
        }

    }
}

// ---- Philox-4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11) -------------------
__device__ inline void philox4x32_10(uint32_t &c0, uint32_t &c1, uint32_t &c2, uint32_t &c3, uint32_t k0,
                                     uint32_t k1) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r) { k0 += 0x9E3779B9u; k1 += 0xBB67AE85u; }
        const uint32_t lo0 = 0xD2511F53u * c0, hi0 = __umulhi(0xD2511F53u, c0);
        const uint32_t lo1 = 0xCD9E8D57u * c2, hi1 = __umulhi(0xCD9E8D57u, c2);
        const uint32_t n0 = hi1 ^ c1 ^ k0, n2 = hi0 ^ c3 ^ k1;
        c0 = n0; c1 = lo1; c2 = n2; c3 = lo0;
    }
}

// ---- block halos in the fused step kernels ----------------------------------
// LDS of a block-halo step kernel: the block's own particles at [0, BLOCK), its
// outside neighbours after them.  Mixed: the 32-byte mirrors, five blocks a CU
// at HALO_CAP.  FP64: 48 bytes, four blocks at HALO_CAP64.
template <bool MIXED, int CAP>
struct HaloLDS {
    float4 x[CAP], n[CAP];
};
template <int CAP>
struct HaloLDS<false, CAP> {
    // one particle's 48 bytes side by side, three 16-byte reads an entry, as its type
    // record (with 8-byte reads of x and n apart a launch for 3.2 M particles took 360
    // us on average, not 355, for 227,000 29.8, not 29.1; the LDS is active for 35 % of
    // the time, two fifths of that bank conflicts)
    Word2 r[CAP][3];
    __device__ __forceinline__ void get(int l, double (&x)[3], double (&n)[3]) const {
        const Word2 a = r[l][0], b = r[l][1], c = r[l][2];
        x[0] = a.x; x[1] = a.y; x[2] = b.x; n[0] = b.y; n[1] = c.x; n[2] = c.y;
    }
    __device__ __forceinline__ void put(int l, const double (&x)[3], const double (&n)[3]) {
        r[l][0] = Word2{x[0], x[1]}; r[l][1] = Word2{x[2], n[0]}; r[l][2] = Word2{n[1], n[2]};
    }
};

// Mixed walk over a staged halo: 16-bit entries, two per word (local index in
// bits 0-9, the neighbour's type in bits 10-12), rows padded to whole groups of
// HALO_GROUP entries with the particle itself.  w, wn: the row's first two
// words.  Words are loaded two ahead; each entry's mirrors are read from LDS one
// entry ahead of its use, and its pair-type record as soon as its word is in; no
// read is under a branch, behind which the compiler waits for all reads in flight.
// The terms and their order are those of the walk over the 32-bit list.
template <int CAP>
__device__ __forceinline__ void range_halo(int nn, uint32_t w, uint32_t wn, const uint32_t *w16,
                                           const HaloLDS<true, CAP> &L, const PairRec *row, const Anchor &ag,
                                           float4 xi, float4 nf, Acc &out) {
    const int nw = halo_row_words(nn);
    if (nw == 0) return;
    const AnchorI ai = unpack(__float_as_uint(xi.w), ag);
    const double ni[3] = {nf.x, nf.y, nf.z};
    float4 xa = L.x[w & 0x3ffu], na = L.n[w & 0x3ffu];
    // past the row's end its last word is read again (not used)
    if (nw == 1) wn = w;
    for (int m = 0; m < nw; ++m) {
        const uint32_t wc = w;
        w = wn;
        wn = w16[min(m + 2, nw - 1) * BLOCK];
        const uint32_t eb = wc >> 16;
        const float4 xb = L.x[eb & 0x3ffu], nb = L.n[eb & 0x3ffu];
        const PairRec pa = row[(wc >> 10) & 7u];
        pair_rec<false>(ag, ai, xi, ni, xa, na, pa, out);
        xa = L.x[w & 0x3ffu]; na = L.n[w & 0x3ffu];
        const PairRec pb = row[eb >> 10];
        pair_rec<false>(ag, ai, xi, ni, xb, nb, pb, out);
    }
}

// FP64 walk over a staged halo: everything of an entry is read one entry ahead
struct HaloEntry64 {
    double x[3], n[3];
    PairRec64 P;
    template <int CAP>
    __device__ __forceinline__ void load(uint32_t e, const HaloLDS<false, CAP> &L, const PairRec64 *row) {
        L.get((int)(e & 0x3ffu), x, n);
        P = row[(e >> 10) & 7u];
    }
};
template <bool PERIODIC, int CAP>
__device__ __forceinline__ void walk_halo64(int nw, uint32_t w, uint32_t wn, const uint32_t *w16,
                                            const HaloLDS<false, CAP> &L, const PairRec64 *row, const Anchor &ag,
                                            const double (&xi)[3], const double (&ni)[3], Acc &acc) {
    auto eval = [&](const HaloEntry64 &q) {
        double X = xi[0] - q.x[0], Y = xi[1] - q.x[1], Z = xi[2] - q.x[2];
        if (PERIODIC) image(ag, X, Y, Z);
        pair_term(q.P, X, Y, Z, ni, q.n[0], q.n[1], q.n[2], acc);
    };
    HaloEntry64 a, b;
    a.load(w, L, row);
    // past the row's end its last word is read again (not used)
    if (nw == 1) wn = w;
    for (int m = 0; m < nw; ++m) {
        b.load(w >> 16, L, row);
        w = wn;
        wn = w16[min(m + 2, nw - 1) * BLOCK];
        eval(a);
        a.load(w, L, row);
        eval(b);
    }
}
template <int CAP>
__device__ __forceinline__ void range_halo(int nn, uint32_t w, uint32_t wn, const uint32_t *w16,
                                           const HaloLDS<false, CAP> &L, const PairRec64 *row, const Anchor &ag,
                                           const double (&xi)[3], const double (&ni)[3], Acc &acc) {
    const int nw = halo_row_words(nn);
    if (nw == 0) return;
    // the box is the same for all: tested here, not at every entry, and no read is under
    // a branch (57 blocks 13.6 -> 13.0 us a launch, 217 Nose-Hoover 15.2 -> 14.5; nothing on
    // 3.2 M particles, whose waves cover for each other)
    if (is_periodic(ag)) walk_halo64<true>(nw, w, wn, w16, L, row, ag, xi, ni, acc);
    else walk_halo64<false>(nw, w, wn, w16, L, row, ag, xi, ni, acc);
}

// What a step kernel's epilogue reads of its particle: all loads issued
// together, before the bonds and ahead of every store (behind the stores, which
// the compiler must take to overlap them, each would wait on its own).
struct StepState {
    double x[3], n[3], v[3], o[3];
};

// Forces of the fused steps: staged halo, or the 32-bit list (no halos, or one
// that does not fit).  Every thread of the block calls it; afterwards i is the
// particle of this lane (the block's lane order when the halo is staged, else
// the lane's own place), ti its type, st its state and acc its forces if
// i < a.n.  False: the step is skipped (`skip`, the same for the whole grid).
//
// A block's time goes to the loads it waits for as much as to the walk, so
// these go out together: everything that depends on the block and lane alone
// (counts, outside neighbours, lane order, row length, the row's first words,
// the own mirrors) at once, then the neighbours' mirrors, and after the walk
// the whole state at once: 434 -> 411 us a launch on 3.2 M particles in mixed
// precision, with the leaner FP64 term (pair_term) 567 -> 405 us in FP64 (averages
// with the launches that find the list spent).  With what came after, a step that
// runs takes 459 us of 479 before, in FP64 423 of 628.
// `spare`: BLOCK doubles of LDS that are free once every thread of the block has
// returned (a barrier lies between).
// `share` runs before the barrier, with its own loads still to come back.
template <bool MIXED, bool HALO, int CAP, typename Skip, typename Share>
__device__ __forceinline__ bool step_forces(const StepArgs &a, const Anchor &ag, long long blk, Skip skip, Share share,
                                            bool &staged, long long &i, int &ti, StepState &st, Acc &acc,
                                            double *&spare) {
    __shared__ typename std::conditional<MIXED, PairRec, PairRec64>::type recs[NT * NT];
    __shared__ BondTab<typename std::conditional<MIXED, float, double>::type> bt;
    __shared__ HaloLDS<MIXED, HALO ? CAP : 1> L;
    spare = reinterpret_cast<double *>(&L);
    const long long col = blk * BLOCK + threadIdx.x;
    constexpr int EXT = HALO ? (CAP - BLOCK + BLOCK - 1) / BLOCK : 1;
    uint32_t hcnt = HALO_OVERFLOW, info = threadIdx.x, w = 0u, wn = 0u, ext[EXT];
    const uint32_t *w16 = nullptr;
    typename std::conditional<MIXED, float4, double[3]>::type xo, no;
    const long long own = col < a.n ? col : blk * BLOCK;
    if constexpr (HALO) {
        hcnt = a.halo_cnt[blk];
        // ext holds HALO_EXT_MAX entries a block; those past hcnt are not used
#pragma unroll
        for (int u = 0; u < EXT; ++u) {
            const int q = u * BLOCK + (int)threadIdx.x;
            ext[u] = a.halo_ext[blk * HALO_EXT_MAX + (q < HALO_EXT_MAX ? q : 0)];
        }
        info = a.hinfo[col];
        w16 = a.nbr16 + list_base(col, a.words);
        w = w16[0];
        wn = w16[BLOCK];
        if constexpr (MIXED) {
            xo = a.pq_in[own].x; no = a.pq_in[own].n;
        } else {
#pragma unroll
            for (int d = 0; d < 3; ++d) { xo[d] = a.x_in[3 * own + d]; no[d] = a.n_in[3 * own + d]; }
        }
    }
    if (skip()) return false;
    staged = HALO && hcnt != HALO_OVERFLOW;
    load_pair_recs(recs);
    load_bonds(bt);
    if constexpr (HALO) {
        if (staged) {
            const int t = (int)threadIdx.x;
            // past the halo's count a lane reads its own record again and drops it
            if constexpr (MIXED) {
                float4 xe[EXT], ne[EXT];
#pragma unroll
                for (int u = 0; u < EXT; ++u) {
                    const PQ &q = a.pq_in[(uint32_t)(u * BLOCK + t) < hcnt ? (long long)ext[u] : own];
                    xe[u] = q.x; ne[u] = q.n;
                }
                L.x[t] = xo; L.n[t] = no;
#pragma unroll
                for (int u = 0; u < EXT; ++u) {
                    const int q = u * BLOCK + t;
                    if ((uint32_t)q < hcnt) { L.x[BLOCK + q] = xe[u]; L.n[BLOCK + q] = ne[u]; }
                }
            } else {
                double xe[EXT][3], ne[EXT][3];
#pragma unroll
                for (int u = 0; u < EXT; ++u) {
                    const long long j = (uint32_t)(u * BLOCK + t) < hcnt ? (long long)ext[u] : own;
#pragma unroll
                    for (int d = 0; d < 3; ++d) { xe[u][d] = a.x_in[3 * j + d]; ne[u][d] = a.n_in[3 * j + d]; }
                }
                L.put(t, xo, no);
#pragma unroll
                for (int u = 0; u < EXT; ++u) {
                    const int q = u * BLOCK + t;
                    if ((uint32_t)q < hcnt) L.put(BLOCK + q, xe[u], ne[u]);
                }
            }
        }
    }
    share();
    __syncthreads();
    const int l = staged ? (int)(info & 0xffu) : (int)threadIdx.x;
    i = blk * BLOCK + l;
    ti = 0;
    if (i >= a.n) return true;
    if constexpr (HALO) {
        if (staged) {
            if constexpr (MIXED) {
                const float4 xi = L.x[l], ni = L.n[l];
                ti = __float_as_int(ni.w);
                range_halo<CAP>((int)(info >> 8), w, wn, w16, L, recs + ti * NT, ag, xi, ni, acc);
            } else {
                double xi[3], ni[3];
                L.get(l, xi, ni);
                ti = a.type[i];
                range_halo<CAP>((int)(info >> 8), w, wn, w16, L, recs + ti * NT, ag, xi, ni, acc);
                finish(ni, acc);
                for (int d = 0; d < 3; ++d) { st.x[d] = xi[d]; st.n[d] = ni[d]; }
            }
        }
    }
    if (!staged) {
        ti = a.type[i];
        // beside a staged walk one neighbour at a time, within its registers
        if constexpr (MIXED) pairs_mixed<false, HALO ? 1 : UNROLL_MIXED>(i, a.kmax, a.pq_in, a.nbr, a.nnbr, ag, recs, acc);
        else pairs_fp64(i, a.kmax, a.x_in, a.n_in, a.type, a.nbr, a.nnbr, ag, recs, acc);
    }
    const int nb = a.has_bonds ? (int)a.nbnd[i] : 0;
    if (MIXED || !staged)
        for (int d = 0; d < 3; ++d) { st.x[d] = a.x_in[3 * i + d]; st.n[d] = a.n_in[3 * i + d]; }
    for (int d = 0; d < 3; ++d) { st.v[d] = a.v[3 * i + d]; st.o[d] = a.o[3 * i + d]; }
    if constexpr (MIXED) bonds_mixed<false>(i, nb, a.stride, a.pq_in, a.bnd, ag, bt, acc);
    else bonds_fp64(i, nb, a.stride, a.x_in, a.bnd, ag, bt, acc);
    return true;
}

// ---- fused timestep: forces + bonds + verlet_langevin ---------------------
// src/openrbc.cpp:219-233 (compute_pairwise_fused, compute_bonded,
// integrate(verlet_langevin)) in one pass; the Langevin update restates
// src/integrate_langevin.h:275-297 in FP64 with counter-based noise.
// HALO: the block's neighbours are staged in LDS from its halo (k_halo) and the
// list is walked as 16-bit local indices; a block marked HALO_OVERFLOW gathers
// from the 32-bit list.
template <bool MIXED, bool HALO, int CAP = MIXED ? HALO_CAP : HALO_CAP64>
__device__ __forceinline__ void step_langevin(const StepArgs &a) {
    // the anchor grid from its device copy (rewritten at every neighbour
    // rebuild, so a captured batch stays valid), a uniform load at the top
    const Anchor ag = *a.anc_dev;
    const unsigned long long step = (a.step0 ? *a.step0 : 0ull) + a.step;
    const int k3 = (int)(step % 3ull);
    const long long blk = block_index(a.swizzle);
    bool staged;
    long long i;
    int ti;
    StepState st;
    Acc acc;
    double *spare;
    auto skip = [&] {
        // skin flag of this step's input positions; no block of this launch writes it
        if (*a.stop || a.dslot[(k3 + 2) % 3] != 0u) {
            if (blockIdx.x == 0 && threadIdx.x == 0) *a.stop = 1;
            return true;
        }
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            a.dslot[(k3 + 1) % 3] = 0u;
            atomicAdd(a.done, 1);
        }
        return false;
    };
    // volume push from the partial sums of the volume, in the order of k_volume_force
    __shared__ double s_push;
    const bool sums_push = a.vol_partial != nullptr;
    double vol = 0.0;
    if (sums_push && (int)threadIdx.x < a.vol_parts) vol = a.vol_partial[threadIdx.x];
    auto share = [&] {
        if (!sums_push || threadIdx.x >= 64) return;
        for (int off = 32; off > 0; off >>= 1) vol += __shfl_xor(vol, off, 64);
        if (threadIdx.x == 0) s_push = a.vol_strength * (a.vol_target - vol) / a.vol_target;
    };
    if (!step_forces<MIXED, HALO, CAP>(a, ag, blk, skip, share, staged, i, ti, st, acc, spare)) return;
    float d2 = 0.f;
    bool bad = false;
    if (i < a.n) {
        const uint32_t wi = a.anc[i], id = a.id[i];
        const float rb[3] = {a.rb[3 * i], a.rb[3 * i + 1], a.rb[3 * i + 2]};
        const double gam = a.gamma[ti], sig = a.sig_group ? a.sig_group[a.grp[i] * NT + ti] : a.sigma[ti];
        double fx = acc.fx, fy = acc.fy, fz = acc.fz;
        const double tx = acc.tx, ty = acc.ty, tz = acc.tz;
        if (a.push || sums_push) {
            // constrain_volume push along the particle's cell normal (src/constrain_volume.h:67-75)
            const int kc = a.aff[i];
            if (kc >= 0) {
                const double sp = (sums_push ? s_push : *a.push) * c_ffd.mass[ti];
                fx += sp * a.cell_normal[3 * kc]; fy += sp * a.cell_normal[3 * kc + 1]; fz += sp * a.cell_normal[3 * kc + 2];
            }
        }
        // rotation: t = n x t; o += dt t; n = normalize(n + (o x n) dt)
        const double nx = st.n[0], ny = st.n[1], nz = st.n[2];
        double ox = st.o[0], oy = st.o[1], oz = st.o[2];
        const double dt = a.dt;
        const double qx = ny * tz - nz * ty, qy = nz * tx - nx * tz, qz = nx * ty - ny * tx;
        ox += dt * qx; oy += dt * qy; oz += dt * qz;
        double gx = nx + (oy * nz - oz * ny) * dt;
        double gy = ny + (oz * nx - ox * nz) * dt;
        double gz = nz + (ox * ny - oy * nx) * dt;
        const double gs = rsqrt(gx * gx + gy * gy + gz * gz);
        gx *= gs; gy *= gs; gz *= gs;
        // translation with uniform [-1,1) noise (src/integrate_langevin.h:282-296)
        uint32_t c0 = id, c1 = (uint32_t)step, c2 = (uint32_t)(step >> 32), c3 = 0u;
        philox4x32_10(c0, c1, c2, c3, (uint32_t)a.seed, (uint32_t)(a.seed >> 32));
        const double u = 4.656612873077392578125e-10;
        const double rx = (double)c0 * u - 1.0, ry = (double)c1 * u - 1.0, rz = (double)c2 * u - 1.0;
        double vx = st.v[0], vy = st.v[1], vz = st.v[2];
        fx -= gam * vx + sig * rx;
        fy -= gam * vy + sig * ry;
        fz -= gam * vz + sig * rz;
        const double dtm = dt * c_ffd.inv_mass[ti];
        vx += fx * dtm; vy += fy * dtm; vz += fz * dtm;
        const double px = st.x[0] + vx * dt, py = st.x[1] + vy * dt, pz = st.x[2] + vz * dt;
        a.x_out[3 * i] = px; a.x_out[3 * i + 1] = py; a.x_out[3 * i + 2] = pz;
        a.n_out[3 * i] = gx; a.n_out[3 * i + 1] = gy; a.n_out[3 * i + 2] = gz;
        a.v[3 * i] = vx; a.v[3 * i + 1] = vy; a.v[3 * i + 2] = vz;
        a.o[3 * i] = ox; a.o[3 * i + 1] = oy; a.o[3 * i + 2] = oz;
        // FP32 mirror with the build-time anchor, and the skin check
        const AnchorI ai = unpack(wi, ag);
        const float r0 = __double2float_rn(px - anchor_pos(ag, 0, ai.x));
        const float r1 = __double2float_rn(py - anchor_pos(ag, 1, ai.y));
        const float r2 = __double2float_rn(pz - anchor_pos(ag, 2, ai.z));
        if (MIXED) {
            PQ q;
            q.x = make_float4(r0, r1, r2, __uint_as_float(wi));
            q.n = make_float4(__double2float_rn(gx), __double2float_rn(gy), __double2float_rn(gz), __int_as_float(ti));
            a.pq_out[i] = q;
        }
        const float e0 = r0 - rb[0], e1 = r1 - rb[1], e2 = r2 - rb[2];
        d2 = e0 * e0 + e1 * e1 + e2 * e2;
        bad = !(isfinite(px) && isfinite(py) && isfinite(pz) && isfinite(gx));
        if (bad) d2 = 3.0e38f;
    }
    // one atomic per wave, and only when some lane moved past its budget:
    // skin/2, or for a particle without list entries the budget k_budget gave it
    bool past = d2 > a.half_skin2;
    if (past && a.bud2 && !bad && a.nnbr[i] == 0) past = d2 > a.bud2[i];
    const unsigned long long over = __ballot(past);
    if (over && __lane_id() == (int)__ffsll((long long)over) - 1) atomicOr(a.dslot + k3, 1u);
    if (bad) atomicOr(a.bad, 1u);
}

template <bool MIXED>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(4))) void k_step_langevin(StepArgs a) {
    step_langevin<MIXED, false>(a);
}
// block halos: 5 blocks of 256 per CU's LDS (96 registers)
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(5))) void k_step_langevin_halo(StepArgs a) {
    step_langevin<true, true>(a);
}
// FP64 halo: 48-byte records, 4 blocks of 256 per CU's LDS
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(4))) void k_step_langevin64_halo(StepArgs a) { step_langevin<false, true>(a); }
// wide halos (HALO_CAP_WIDE local indices): the mixed kernel at 4 blocks of
// 256 per CU (128 registers), the FP64 one at 3
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(4))) void k_step_langevin_halo_wide(StepArgs a) {
    step_langevin<true, true, HALO_CAP_WIDE>(a);
}
__global__ __launch_bounds__(BLOCK) void k_step_langevin64_halo_wide(StepArgs a) {
    step_langevin<false, true, HALO_CAP_WIDE>(a);
}

// ---- fused forces + post_toque_final_update (NH second half) --------------
// src/integrate_nh.h:237-273 after compute_pairwise_fused/compute_bonded, in
// the arithmetic of the unfused pair k_forces + k_nh_second: the mixed sums
// are rounded to FP32 as the FP32 force arrays hold them; t = n x t;
// v += dt/2 (f/m - zeta v); o += dt/2 t; f and n x t stored (FP32 arrays in
// mixed precision) for the next first half; KE partial per particle block.
template <bool MIXED, bool HALO, int CAP = MIXED ? HALO_CAP : HALO_CAP64>
__device__ __forceinline__ void step_nh_second(const StepArgs &a, float *f32, float *t32, double *f64, double *t64,
                                               double *ke_partial, const ZetaUp &zup) {
    const long long blk = block_index(a.swizzle);
    bool staged;
    long long i;
    int ti;
    StepState st;
    Acc acc;
    double *spare;
    auto skip = [&] {
        if (!a.nh_gate) return false;
        // batched run: the first half of this step found a particle past its
        // budget (slot step % 3), or an earlier step stopped: nothing to do
        const int k3 = (int)(a.step % 3ull);
        if (*a.stop || a.dslot[k3] != 0u) {
            if (blockIdx.x == 0 && threadIdx.x == 0) *a.stop = 1;
            return true;
        }
        if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(a.done, 1);
        return false;
    };
    __shared__ double ws_zeta[ZETA_PARTS / 64];
    auto share = [&] {
        if (zup.nb > 0) zeta_sums(zup, ws_zeta);
    };
    if (!step_forces<MIXED, HALO, CAP>(a, a.anc_grid, blk, skip, share, staged, i, ti, st, acc, spare)) return;
    const double zeta = zup.nb > 0 ? zeta_now(zup, ws_zeta) : *zup.in;
    double ke = 0.0;
    if (i < a.n) {
        double f[3], t[3];
        if constexpr (MIXED) {
            f[0] = (float)acc.fx; f[1] = (float)acc.fy; f[2] = (float)acc.fz;
            t[0] = (float)acc.tx; t[1] = (float)acc.ty; t[2] = (float)acc.tz;
        } else {
            f[0] = acc.fx; f[1] = acc.fy; f[2] = acc.fz;
            t[0] = acc.tx; t[1] = acc.ty; t[2] = acc.tz;
        }
        const double m = c_ffd.mass[ti];
        double v[3], q[3];
        const double (&n)[3] = st.n;
        for (int d = 0; d < 3; ++d) v[d] = st.v[d];
        q[0] = n[1] * t[2] - n[2] * t[1];
        q[1] = n[2] * t[0] - n[0] * t[2];
        q[2] = n[0] * t[1] - n[1] * t[0];
        for (int d = 0; d < 3; ++d) {
            v[d] += 0.5 * a.dt * (f[d] / m - zeta * v[d]);
            a.o[3 * i + d] = st.o[d] + 0.5 * a.dt * q[d];
            a.v[3 * i + d] = v[d];
        }
        if constexpr (MIXED) {
            for (int d = 0; d < 3; ++d) { f32[3 * i + d] = (float)f[d]; t32[3 * i + d] = (float)q[d]; }
        } else {
            for (int d = 0; d < 3; ++d) { f64[3 * i + d] = f[d]; t64[3 * i + d] = q[d]; }
        }
        ke = 0.5 * m * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    }
    if constexpr (HALO) {
        // back to particle order, the order of the unfused reduction
        if (staged) {                         // block-uniform
            __syncthreads();
            spare[i - blk * BLOCK] = ke;
            __syncthreads();
            ke = spare[threadIdx.x];
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) ke += __shfl_xor(ke, off, 64);
    __shared__ double ws[BLOCK / 64];
    if (__lane_id() == 0) ws[threadIdx.x >> 6] = ke;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0;
        for (int w = 0; w < BLOCK / 64; ++w) s += ws[w];
        ke_partial[blk] = s;          // by particle block, the order of the unfused reduction
    }
}

template <bool MIXED>
__global__ __launch_bounds__(BLOCK) void k_step_nh_second(StepArgs a, float *f32, float *t32, double *f64,
                                                          double *t64, double *ke_partial, ZetaUp zup) {
    step_nh_second<MIXED, false>(a, f32, t32, f64, t64, ke_partial, zup);
}
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(5))) void k_step_nh_second_halo(StepArgs a, float *f32, float *t32,
                                                                              double *f64, double *t64,
                                                                              double *ke_partial,
                                                                              ZetaUp zup) {
    step_nh_second<true, true>(a, f32, t32, f64, t64, ke_partial, zup);
}
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(4))) void k_step_nh_second64_halo(StepArgs a, float *f32, float *t32, double *f64,
                                                                 double *t64, double *ke_partial,
                                                                 ZetaUp zup) {
    step_nh_second<false, true>(a, f32, t32, f64, t64, ke_partial, zup);
}
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(4))) void k_step_nh_second_halo_wide(
    StepArgs a, float *f32, float *t32, double *f64, double *t64, double *ke_partial, ZetaUp zup) {
    step_nh_second<true, true, HALO_CAP_WIDE>(a, f32, t32, f64, t64, ke_partial, zup);
}
__global__ __launch_bounds__(BLOCK) void k_step_nh_second64_halo_wide(StepArgs a, float *f32, float *t32,
                                                                      double *f64, double *t64, double *ke_partial,
                                                                      ZetaUp zup) {
    step_nh_second<false, true, HALO_CAP_WIDE>(a, f32, t32, f64, t64, ke_partial, zup);
}

inline unsigned nblk(long long n) { return (unsigned)((n + BLOCK - 1) / BLOCK); }

}  // namespace

void upload_ff(const FFTab<double> &d, const FFTab<float> &f, hipStream_t s) {
    ORBC_HIP_CHECK(hipMemcpyToSymbolAsync(HIP_SYMBOL(c_ffd), &d, sizeof(d), 0, hipMemcpyHostToDevice, s));
    ORBC_HIP_CHECK(hipMemcpyToSymbolAsync(HIP_SYMBOL(c_fff), &f, sizeof(f), 0, hipMemcpyHostToDevice, s));
    upload_mass(d.mass, s);
    ORBC_HIP_CHECK(hipStreamSynchronize(s));
}

void launch_forces(const ForceArgs &a, bool mixed, bool energy, bool pair, bool bond, hipStream_t s) {
    if (a.n <= 0) return;
    const dim3 g(nblk(a.n)), b(BLOCK);
    if (mixed) {
        if (energy) hipLaunchKernelGGL((k_forces<true, true>), g, b, 0, s, a, (int)pair, (int)bond);
        else hipLaunchKernelGGL((k_forces<true, false>), g, b, 0, s, a, (int)pair, (int)bond);
    } else {
        if (energy) hipLaunchKernelGGL((k_forces<false, true>), g, b, 0, s, a, (int)pair, (int)bond);
        else hipLaunchKernelGGL((k_forces<false, false>), g, b, 0, s, a, (int)pair, (int)bond);
    }
}

void launch_step_langevin(const StepArgs &a, bool mixed, hipStream_t s) {
    if (a.n <= 0) return;
    const dim3 g(nblk(a.n)), b(BLOCK);
    const bool wide = a.halo_cap == HALO_CAP_WIDE;
    if (mixed && a.halo_cnt && wide) hipLaunchKernelGGL(k_step_langevin_halo_wide, g, b, 0, s, a);
    else if (mixed && a.halo_cnt) hipLaunchKernelGGL(k_step_langevin_halo, g, b, 0, s, a);
    else if (mixed) hipLaunchKernelGGL(k_step_langevin<true>, g, b, 0, s, a);
    else if (a.halo_cnt && wide) hipLaunchKernelGGL(k_step_langevin64_halo_wide, g, b, 0, s, a);
    else if (a.halo_cnt) hipLaunchKernelGGL(k_step_langevin64_halo, g, b, 0, s, a);
    else hipLaunchKernelGGL(k_step_langevin<false>, g, b, 0, s, a);
}

void launch_step_nh_second(const StepArgs &a, bool mixed, float *f32, float *t32, double *f64, double *t64,
                           double *ke_partial, const ZetaUp &zeta, hipStream_t s) {
    if (a.n <= 0) return;
    const dim3 g(nblk(a.n)), b(BLOCK);
    const bool wide = a.halo_cap == HALO_CAP_WIDE;
    if (mixed && a.halo_cnt && wide)
        hipLaunchKernelGGL(k_step_nh_second_halo_wide, g, b, 0, s, a, f32, t32, f64, t64, ke_partial, zeta);
    else if (mixed && a.halo_cnt)
        hipLaunchKernelGGL(k_step_nh_second_halo, g, b, 0, s, a, f32, t32, f64, t64, ke_partial, zeta);
    else if (mixed) hipLaunchKernelGGL(k_step_nh_second<true>, g, b, 0, s, a, f32, t32, f64, t64, ke_partial, zeta);
    else if (a.halo_cnt && wide)
        hipLaunchKernelGGL(k_step_nh_second64_halo_wide, g, b, 0, s, a, f32, t32, f64, t64, ke_partial, zeta);
    else if (a.halo_cnt)
        hipLaunchKernelGGL(k_step_nh_second64_halo, g, b, 0, s, a, f32, t32, f64, t64, ke_partial, zeta);
    else hipLaunchKernelGGL(k_step_nh_second<false>, g, b, 0, s, a, f32, t32, f64, t64, ke_partial, zeta);
}

void launch_min_step(const MinArgs &a, bool mixed, hipStream_t s) {
    if (a.s.n <= 0) return;
    const dim3 g(nblk(a.s.n)), b(BLOCK);
    if (mixed) hipLaunchKernelGGL(k_min_step<true>, g, b, 0, s, a);
    else hipLaunchKernelGGL(k_min_step<false>, g, b, 0, s, a);
}

void launch_pairs_export(const ForceArgs &a, bool mixed, unsigned *ids_i, unsigned *ids_j, unsigned long long *count,
                         long long cap, hipStream_t s) {
    if (a.n <= 0) return;
    const dim3 g(nblk(a.n)), b(BLOCK);
    if (mixed) hipLaunchKernelGGL(k_pairs_export<true>, g, b, 0, s, a, ids_i, ids_j, count, cap);
    else hipLaunchKernelGGL(k_pairs_export<false>, g, b, 0, s, a, ids_i, ids_j, count, cap);
}

}  // namespace orbc
