// sg_direct.hip -- the O(N^2) pair kernels for gfx950 (CDNA4).
//
// Reference: dev_compute_forces<256> and dev_force_ij_nkernel{0,1,2}
// (pbe/src/SPHgrav_lib2/grav_force_direct.cu:55-502): one i per thread, j in
// 256-wide shared-memory tiles, every pair through the full three-way softened
// branch, float-float (Fast2Sum) accumulation of every term.
//
// Whole sets and batches take their far pairs from sg_sym.hip / sg_sym64.hip;
// here are the visits these leave (k_sym_rest), the wave-sized work items of
// small i-ranges (k_pair_wave), the grad-h term alone (k_psi_only) and the
// ordered tile kernels, which run for explicit tile shapes, large parts of a
// set and small FP64 sets.
//
// Design of the ordered tile kernels (wave64, VALU-bound):
//   * particles arrive sorted along a Morton curve (sg_prep.hip), so an
//     i-group of 64*IPL consecutive particles (one wave) and a j-tile of TJ
//     consecutive particles (four chunks of TC) are both spatially compact;
//   * each wave holds IPL i-particles per lane in registers and classifies
//     every (wave, tile) and then every (wave, chunk) with box tests and a
//     per-lane test (near_mask): a far chunk has every pair Newtonian (the
//     grav_force_direct.cu:69-75 branch) and runs a branch-free body of 13
//     VALU operations plus one v_rsq_f32 per pair;
//   * j data is staged through LDS per workgroup as FP32 {x_hi, y_hi, z_hi, m}
//     and as FP64 {x, y, z} relative to an FP64 origin taken per workgroup,
//     written from coalesced FP64 global loads and read back as same-address
//     (broadcast) LDS reads.  Chunks use hi-only differences, except those
//     nearer to the wave's box than WIDE_K times its largest |x_i - O|,
//     which form the difference in FP64 and round it once;
//   * FP32 partial sums over FOLD j are folded into FP64 accumulators (the
//     cross-tile and cross-partition reductions are FP64);
//   * near chunks (pairs that may be softened) are listed per wave and run
//     after its far loop in the wave's own LDS slice: FP64-formed
//     differences, the FP32 body for the Newtonian lanes, FP64 near_pair for
//     the softened ones, each lane walking its own list of them (the
//     Wendland polynomials carry coefficients up to 9009 that cancel to O(1)
//     near q = 1, which FP32 cannot resolve);
//   * the FP64 comparison pass and the grad-h pass flag near chunks for a
//     separate near kernel instead;
//   * REDUCE kernel: fixed-order FP64 sum over j-partitions, scattered back to
//     input order.
//
// Two launch forms share the block-level code: one particle set (grid over
// i-blocks x j-partitions), and a batch of independent sets in one persistent
// launch whose workgroups pull (set, i-block, j-partition) items from a
// queue.
#include "sg_internal.h"
#include "sg_device.h"

#include <math.h>

namespace sg {
namespace {

constexpr int TS = 128;                 // j per LDS stage; TJ / TS stages per tile
constexpr int FOLD = 32;                // FP32 partial sums span FOLD j
constexpr int NEAR_WAVES = 4;           // waves sharing one group's near tiles

static_assert(TJ % TS == 0, "tile must be a whole number of stages");
static_assert(TS % TC == 0 && TC % FOLD == 0, "stage = whole chunks = whole folds");

// The part of a launch one far-kernel workgroup works on.
struct Block {
    int64_t ibase;          // first (sorted) i of the workgroup
    int64_t iend;           // end of the i segment the block lies in
    int t0, t1, tstep;      // j-tiles t0, t0 + tstep, ... below t1
    int fbase;              // near flags are indexed by t - fbase
    unsigned char *flags;   // near flags of the workgroup's first wave, [t - fbase]
    int64_t fstride;        // flag stride between consecutive waves
    double *part;           // partial sums: part[c * pstride + i], c = ax, ay, az, pot
    int64_t pstride;
};

// The part of a launch one near-kernel workgroup works on (one i-group).
struct Group {
    int64_t gbase, iend;
    int t0, t1;
    const unsigned char *flags;   // [t - t0]
    double *part;
    int64_t pstride;
    double *psipart;              // psi partial sums of this j-partition (PSI kernels)
};

// ------------------------------------------------ far block, FP32 + comp.
// One Newtonian pair (i <- j) in FP32 from its difference dr and m_j.  FIRST
// starts the partial sums (the first j of a fold writes them, which saves
// clearing them).
template <bool FIRST>
__device__ __forceinline__ void far_pair_fp32(float dx, float dy, float dz, float mj, float &fx,
                                              float &fy, float &fz, float &fp)
{
    const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
    const float ri = __builtin_amdgcn_rsqf(r2);
    const float mr = mj * ri;
    const float mr3 = mr * ri * ri;
    if (FIRST) {
        fx = mr3 * dx;
        fy = mr3 * dy;
        fz = mr3 * dz;
        fp = mr;
    } else {
        fx = fmaf(mr3, dx, fx);
        fy = fmaf(mr3, dy, fy);
        fz = fmaf(mr3, dz, fz);
        fp += mr;
    }
}

// m_j travels in the FP64 stage as the low half of the w slot.
__device__ __forceinline__ double pack_mass(float m)
{
    const float2 v = make_float2(m, 0.0f);
    return __builtin_bit_cast(double, v);
}

// The difference of one pair for the FP32 body.  Far tiles use hi-only
// differences (x_j,hi - x_i,hi).  WIDE tiles (close relative to the wave's
// spread about the origin) form x_j - x_i in FP64 from the FP64 stage and
// round it once (two ops per axis): exact to half an ulp of r, with no
// shared error from the rounding of x_i.
template <bool WIDE>
__device__ __forceinline__ void far_diff(const float4 *ph, const double4 *pd, int jj, float xh,
                                         float yh, float zh, double xr, double yr, double zr,
                                         float &dx, float &dy, float &dz, float &mj)
{
    if (WIDE) {
        const double4 q = pd[jj];
        dx = (float)(q.x - xr);
        dy = (float)(q.y - yr);
        dz = (float)(q.z - zr);
        mj = __builtin_bit_cast(float2, q.w).x;
    } else {
        const float4 p = ph[jj];
        dx = p.x - xh;
        dy = p.y - yh;
        dz = p.z - zh;
        mj = p.w;
    }
}

// One chunk (TC j) of far pairs from LDS.  The FOLD j of a fold are
// unrolled, so the LDS reads use immediate offsets from one address per fold.
template <int IPL, bool WIDE>
__device__ __forceinline__ void far_chunk_fp32(const float4 *s_hi, const double4 *s_p,
                                               const float (&xh)[IPL], const float (&yh)[IPL],
                                               const float (&zh)[IPL], const double (&xr)[IPL],
                                               const double (&yr)[IPL], const double (&zr)[IPL],
                                               double (&ax)[IPL], double (&ay)[IPL],
                                               double (&az)[IPL], double (&ap)[IPL])
{
#pragma unroll 1
    for (int j0 = 0; j0 < TC; j0 += FOLD) {
        const float4 *ph = s_hi + j0;
        const double4 *pd = s_p + j0;
        float fx[IPL], fy[IPL], fz[IPL], fp[IPL];
#pragma unroll
        for (int k = 0; k < IPL; ++k) {
            float dx, dy, dz, mj;
            far_diff<WIDE>(ph, pd, 0, xh[k], yh[k], zh[k], xr[k], yr[k], zr[k], dx, dy, dz, mj);
            far_pair_fp32<true>(dx, dy, dz, mj, fx[k], fy[k], fz[k], fp[k]);
        }
#pragma unroll
        for (int jj = 1; jj < FOLD; ++jj) {
#pragma unroll
            for (int k = 0; k < IPL; ++k) {
                float dx, dy, dz, mj;
                far_diff<WIDE>(ph, pd, jj, xh[k], yh[k], zh[k], xr[k], yr[k], zr[k], dx, dy, dz,
                               mj);
                far_pair_fp32<false>(dx, dy, dz, mj, fx[k], fy[k], fz[k], fp[k]);
            }
        }
#pragma unroll
        for (int k = 0; k < IPL; ++k) {
            ax[k] += (double)fx[k];
            ay[k] += (double)fy[k];
            az[k] += (double)fz[k];
            ap[k] -= (double)fp[k];
        }
    }
}

// One side k of a softened pair: adds F(r,H_k) and P(r,H_k) (without m_j).
// The kernel choice NK is a template parameter of the near kernels: with one
// polynomial per instantiation the register footprint drops by a third.
// With PSI it also adds P(q) + q^2 A(q) to *ps when the side is softened: the
// grad-h term's dphidh(2q) = -(P(q) + q^2 A(q))/2 (kernels.f:215-279).
template <int NK, bool PSI = false>
__device__ __forceinline__ void soft_side(double r, double ri, double r2, double H,
                                          double invH, double &gacc, double &gpot,
                                          double *ps = nullptr)
{
    if (r2 <= H * H) {
        const double q = r * invH;
        double A, P;
        poly_AP(NK, q, H * ri, A, P);
        gacc += A * invH * invH * invH;
        gpot += P * invH;
        if (PSI) *ps = fma(q * q, A, P);
    } else {
        gacc += ri * ri * ri;
        gpot -= ri;
    }
}

// Ordered pair (i <- j), FP64, the semantics of grav_force_direct.cu:55-396
// with the r == 0 rule documented in include/sphgrav.h.
// With PSI, ps accumulates m_j (P(q_i) + q_i^2 A(q_i)) over the pairs with
// r <= H_i (the grad-h softening sum before its -2/H_i^2 factor).
// The j side's 1/H_j and H_j^2 come precomputed from the LDS stage (one
// division per staged particle instead of one per pair).
template <bool FAST, int NK, bool PSI = false>
__device__ __forceinline__ void near_pair(double dx, double dy, double dz, double Hi,
                                          double invHi, double hi2, double Hj, double invHj,
                                          double hj2, double mj, bool gasj, bool same,
                                          double &ax, double &ay, double &az, double &ap,
                                          double *ps = nullptr)
{
    const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
    if (r2 >= fmax(hi2, hj2)) {
        const double ri = rsqrt64<FAST>(r2);
        const double mr = mj * ri;
        const double mr3 = mr * ri * ri;
        ax = fma(mr3, dx, ax);
        ay = fma(mr3, dy, ay);
        az = fma(mr3, dz, az);
        ap -= mr;
    } else if (r2 == 0.0) {
        if (!same || gasj) ap -= self_coeff(NK) * mj * (invHi + invHj);
        if (PSI) *ps -= 2.0 * self_coeff(NK) * mj;   // P(0) = -2c
    } else {
        const double ri = rsqrt64<FAST>(r2);
        const double r = r2 * ri;
        double gacc = 0.0, gpot = 0.0;
        double psk = 0.0;
        soft_side<NK, PSI>(r, ri, r2, Hi, invHi, gacc, gpot, &psk);
        soft_side<NK>(r, ri, r2, Hj, invHj, gacc, gpot);
        if (PSI) *ps = fma(mj, psk, *ps);
        const double hm = 0.5 * mj;
        const double f = hm * gacc;
        ax = fma(f, dx, ax);
        ay = fma(f, dy, ay);
        az = fma(f, dz, az);
        ap = fma(hm, gpot, ap);
    }
}

// FP64 i-side softening state of the near pairs.
template <int IPL>
__device__ __forceinline__ void near_i_state(const SortedSet &I, const int64_t (&ii)[IPL],
                                             double (&Hi)[IPL], double (&invHi)[IPL],
                                             double (&hi2)[IPL], int (&idi)[IPL])
{
#pragma unroll
    for (int k = 0; k < IPL; ++k) {
        Hi[k] = fabs(I.Hs[ii[k]]);
        invHi[k] = 1.0 / Hi[k];
        hi2[k] = Hi[k] * Hi[k];
        idi[k] = I.idx[ii[k]];
    }
}

// Per-wave LDS of the fused FP32C far kernel: the wave's list of deferred
// near tiles and the slice a near chunk is staged in.
constexpr int NLIST = 128;   // deferred near tiles per wave (more run at once)
struct NearSlice {
    double4 p[TC];           // x, y, z relative to the origin; w: {FP32 m, FP32 H^2}
    double hs[TC];           // signed H (> 0: gas)
    double hinv[TC];         // 1 / |H|
    double m[TC];
    uint32_t list[NLIST];    // (tile - t0) << 4 | chunk mask
};

// Stages one particle per lane in the wave's slice: its position relative to
// the origin, mass and signed H.  Returns the lanes that hold particles (not
// massless padding).
__device__ __forceinline__ uint64_t near_stage(NearSlice &sl, double rx, double ry, double rz,
                                               double mj, double hs)
{
    const int lane = threadIdx.x & 63;
    const float mh[2] = {(float)mj, (float)(hs * hs)};
    const uint64_t real = __ballot(mj > 0.0);
    wave_lds_sync();
    sl.p[lane] = make_double4(rx, ry, rz, __builtin_bit_cast(double, mh));
    sl.hs[lane] = hs;
    sl.hinv[lane] = 1.0 / fabs(hs);
    sl.m[lane] = mj;
    wave_lds_sync();
    return real;
}

// Evaluates the chunk staged in the slice (particles j0c ..).  Each pair
// difference is formed in FP64 and rounded once to FP32 (two ops per axis;
// near pairs are close, where the hi+lo difference would lose the low bits
// of the i position whenever |x_i - O| < |x_j - O|, an error that does not
// average out over j).  The FP32 body then runs every pair with the lanes
// whose pair may be softened (r^2 < max(H_i^2, H_j^2) in FP32, r = 0
// included) masked out; the j where a lane was masked are recorded in a
// wave-uniform bit mask, and those lanes' pairs then run in FP64 through
// near_pair from the slice, each lane over its own list (a pair is taken by
// exactly one of the two, so a borderline FP32 decision costs only
// rounding).  Wave-local: no block barrier.
template <int IPL, int NK>
__device__ __forceinline__ void near_chunk_eval(
    NearSlice &sl, uint64_t real, const SortedSet &J, int64_t j0c, const double (&xr)[IPL],
    const double (&yr)[IPL], const double (&zr)[IPL], const double (&Hi)[IPL],
    const double (&invHi)[IPL], const double (&hi2)[IPL], const int (&idi)[IPL], double (&ax)[IPL],
    double (&ay)[IPL], double (&az)[IPL], double (&ap)[IPL], unsigned (&nfp64)[IPL])
{
    float hi2f[IPL];
#pragma unroll
    for (int k = 0; k < IPL; ++k) hi2f[k] = (float)hi2[k];
    uint64_t jmask = 0;   // wave-uniform: j with at least one masked lane
#pragma unroll 1
    for (int j0 = 0; j0 < TC; j0 += FOLD) {
        float fx[IPL], fy[IPL], fz[IPL], fp[IPL];
#pragma unroll
        for (int k = 0; k < IPL; ++k) fx[k] = fy[k] = fz[k] = fp[k] = 0.0f;
        for (int jj = j0; jj < j0 + FOLD; ++jj) {
            const double4 p = sl.p[jj];
            const float2 mh = __builtin_bit_cast(float2, p.w);   // m_j, H_j^2
            bool any = false;
#pragma unroll
            for (int k = 0; k < IPL; ++k) {
                const float dx = (float)(p.x - xr[k]);
                const float dy = (float)(p.y - yr[k]);
                const float dz = (float)(p.z - zr[k]);
                const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                const bool soft = r2 < fmaxf(hi2f[k], mh.y);
                const float ri = soft ? 0.0f : __builtin_amdgcn_rsqf(r2);
                const float mr = mh.x * ri;
                const float mr3 = mr * ri * ri;
                fx[k] = fmaf(mr3, dx, fx[k]);
                fy[k] = fmaf(mr3, dy, fy[k]);
                fz[k] = fmaf(mr3, dz, fz[k]);
                fp[k] += mr;
                any = any || soft;
            }
            if (__ballot(any)) jmask |= 1ull << jj;
        }
#pragma unroll
        for (int k = 0; k < IPL; ++k) {
            ax[k] += (double)fx[k];
            ay[k] += (double)fy[k];
            az[k] += (double)fz[k];
            ap[k] -= (double)fp[k];
        }
    }
    // The masked pairs in FP64.  A wave-wide walk over the j of jmask would
    // run near_pair with about one lane in eight active, so the walk only
    // repeats the FP32 decision to give each lane its own list, and each
    // lane then runs its list (the wave takes as many steps as its longest).
    uint64_t own[IPL];
#pragma unroll
    for (int k = 0; k < IPL; ++k) own[k] = 0;
    while (jmask) {
        const int jj = __builtin_ctzll(jmask);
        jmask &= jmask - 1;
        const double4 p = sl.p[jj];
        const float2 mh = __builtin_bit_cast(float2, p.w);
#pragma unroll
        for (int k = 0; k < IPL; ++k) {
            // the same FP32 decision as above
            const float dx = (float)(p.x - xr[k]), dy = (float)(p.y - yr[k]),
                        dz = (float)(p.z - zr[k]);
            const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
            if (r2 < fmaxf(hi2f[k], mh.y)) own[k] |= 1ull << jj;
        }
    }
#pragma unroll
    for (int k = 0; k < IPL; ++k) {
        // the counter covers pairs of particles; padding pairs (m_j = 0,
        // evaluated all the same) are left out
        nfp64[k] += (unsigned)__builtin_popcountll(own[k] & real);
        while (own[k]) {
            const int jj = __builtin_ctzll(own[k]);
            own[k] &= own[k] - 1;
            const double4 p = sl.p[jj];
            const double mj = sl.m[jj], hs = sl.hs[jj], ha = fabs(hs), hinv = sl.hinv[jj];
            const double ddx = p.x - xr[k], ddy = p.y - yr[k], ddz = p.z - zr[k];
            // the self pair only matters at r = 0: the index is read then
            const bool same = ddx == 0.0 && ddy == 0.0 && ddz == 0.0 &&
                              J.idx[j0c + jj] == idi[k];
            near_pair<true, NK>(ddx, ddy, ddz, Hi[k], invHi[k], hi2[k], ha, hinv, ha * ha, mj,
                                hs > 0.0, same, ax[k], ay[k], az[k], ap[k]);
        }
    }
}

// Stages chunk c of tile t and evaluates it.
template <int IPL, int NK>
__device__ __forceinline__ void near_chunk_slice(
    NearSlice &sl, const SortedSet &J, int t, int c, double Ox, double Oy, double Oz,
    const double (&xr)[IPL], const double (&yr)[IPL], const double (&zr)[IPL],
    const double (&Hi)[IPL], const double (&invHi)[IPL], const double (&hi2)[IPL],
    const int (&idi)[IPL], double (&ax)[IPL], double (&ay)[IPL], double (&az)[IPL],
    double (&ap)[IPL], unsigned (&nfp64)[IPL])
{
    const int lane = threadIdx.x & 63;
    const int64_t j = (int64_t)t * TJ + c * TC + lane;
    const uint64_t real = near_stage(sl, J.x[j] - Ox, J.y[j] - Oy, J.z[j] - Oz, J.m[j], J.Hs[j]);
    near_chunk_eval<IPL, NK>(sl, real, J, (int64_t)t * TJ + c * TC, xr, yr, zr, Hi, invHi, hi2, idi,
                             ax, ay, az, ap, nfp64);
}

// FUSED (the forward FP32C pass): the chunks a wave cannot classify as far
// are listed and run by the wave alone after its far loop (in its own LDS
// slice, no block barrier in between, so one wave's near work does not hold
// the others at the stage barriers); a list that fills up runs the rest at
// once.  Not FUSED (the grad-h pass): they are flagged in b.flags for the
// near kernel.
template <int WG, int IPL, int NK, bool FUSED>
__device__ __forceinline__ void far_block_fp32c(const SortedSet &I, const SortedSet &J,
                                                const TileMeta *tiles, const TileMeta *chunks,
                                                const Block &b, unsigned long long *stats,
                                                float4 *s_hi, double4 *s_p, NearSlice *s_near)
{
    constexpr int WI = 64 * IPL;   // i per wave
    constexpr int GI = WG * IPL;   // i per workgroup
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;

    // FP64 origin of this workgroup: its middle i-particle.
    const int64_t io = min(b.ibase + GI / 2, b.iend - 1);
    const double Ox = I.x[io], Oy = I.y[io], Oz = I.z[io];

    float xh[IPL], yh[IPL], zh[IPL], hf[IPL];
    double xr[IPL], yr[IPL], zr[IPL];
    int64_t ii[IPL];
    bool valid[IPL];
    float bl[3] = {INFINITY, INFINITY, INFINITY}, bh[3] = {-INFINITY, -INFINITY, -INFINITY};
    float hmax = 0.0f, reach2 = 0.0f;
#pragma unroll
    for (int k = 0; k < IPL; ++k) {
        const int64_t i = b.ibase + wv * WI + k * 64 + lane;
        valid[k] = i < b.iend;
        ii[k] = valid[k] ? i : b.iend - 1;
        xr[k] = I.x[ii[k]] - Ox;
        yr[k] = I.y[ii[k]] - Oy;
        zr[k] = I.z[ii[k]] - Oz;
        xh[k] = (float)xr[k];
        yh[k] = (float)yr[k];
        zh[k] = (float)zr[k];
        hf[k] = (float)fabs(I.Hs[ii[k]]);
        bl[0] = fminf(bl[0], xh[k]); bl[1] = fminf(bl[1], yh[k]); bl[2] = fminf(bl[2], zh[k]);
        bh[0] = fmaxf(bh[0], xh[k]); bh[1] = fmaxf(bh[1], yh[k]); bh[2] = fmaxf(bh[2], zh[k]);
        hmax = fmaxf(hmax, hf[k]);
        reach2 = fmaxf(reach2, fmaf(xh[k], xh[k], fmaf(yh[k], yh[k], zh[k] * zh[k])));
    }
    for (int c = 0; c < 3; ++c) {
        bl[c] = wave_min(bl[c]);
        bh[c] = wave_max(bh[c]);
    }
    hmax = wave_max(hmax);
    // close chunks take FP64-formed differences: those nearer than WIDE_K
    // times the wave's largest |x_i - O| (Euclidean)
    const float wide_d2 = WIDE_K * WIDE_K * wave_max(reach2) * (1.0f + FAR_MARGIN);

    double ax[IPL], ay[IPL], az[IPL], ap[IPL];
#pragma unroll
    for (int k = 0; k < IPL; ++k) ax[k] = ay[k] = az[k] = ap[k] = 0.0;

    // a wave past the end of its segment (the tail of the last i-block)
    // computes nothing and flags nothing
    const bool active = uniform_i(b.ibase + wv * WI < b.iend) != 0;
    unsigned nearv = 0, widev = 0;   // wave-uniform counts of near and wide chunk visits
    unsigned nfp64[IPL];             // per lane: pairs evaluated in FP64 (near tail)
#pragma unroll
    for (int k = 0; k < IPL; ++k) nfp64[k] = 0;
    int nlist = 0;   // wave-uniform
    unsigned char *flags = b.flags + wv * b.fstride;
    for (int t = b.t0; t < b.t1; t += b.tstep) {
        const TileMeta &tm = tiles[t];
        const float d2 = box_dist2(tm, Ox, Oy, Oz, bl, bh);
        const unsigned mask =
            active ? near_mask<IPL>(chunks, t, tm, d2, Ox, Oy, Oz, bl, bh, hmax, xh, yh, zh, hf)
                   : 0u;
        // chunks of a close tile that are themselves close
        unsigned widem = 0;
        if (uniform_i(d2 < wide_d2) != 0)
            for (int c = 0; c < CHUNKS; ++c)
                if (uniform_i(box_dist2(chunks[(int64_t)t * CHUNKS + c], Ox, Oy, Oz, bl, bh) <
                              wide_d2) != 0)
                    widem |= 1u << c;
        nearv += __builtin_popcount(mask);
        if (active) widev += __builtin_popcount(widem & ~mask);
        bool near_tile_now = false;   // a full list: this tile's near chunks run below
        if (!FUSED) {
            if (lane == 0) flags[t - b.fbase] = (unsigned char)mask;
        } else if (mask) {
            if (nlist < NLIST) {
                if (lane == 0)
                    s_near[wv].list[nlist] = ((uint32_t)((t - b.t0) / b.tstep) << 4) | mask;
                ++nlist;
            } else {
                near_tile_now = true;
            }
        }
        if (FUSED && near_tile_now) {
            double Hi[IPL], invHi[IPL], hi2[IPL];
            int idi[IPL];
            near_i_state<IPL>(I, ii, Hi, invHi, hi2, idi);
            for (int c = 0; c < CHUNKS; ++c)
                if ((mask >> c) & 1u)
                    near_chunk_slice<IPL, NK>(s_near[wv], J, t, c, Ox, Oy, Oz, xr, yr, zr, Hi,
                                              invHi, hi2, idi, ax, ay, az, ap, nfp64);
        }
        if (WG == 64 && mask == (1u << CHUNKS) - 1) continue;
        for (int s = 0; s < TJ / TS; ++s) {
            __syncthreads();
            for (int jj = tid; jj < TS; jj += WG) {
                const int64_t j = (int64_t)t * TJ + s * TS + jj;
                const double rx = J.x[j] - Ox, ry = J.y[j] - Oy, rz = J.z[j] - Oz;
                const float mf = (float)J.m[j];
                s_hi[jj] = make_float4((float)rx, (float)ry, (float)rz, mf);
                s_p[jj] = make_double4(rx, ry, rz, pack_mass(mf));
            }
            __syncthreads();
            if (!active) continue;
            for (int h = 0; h < TS / TC; ++h) {
                const int c = s * (TS / TC) + h;
                if ((mask >> c) & 1u) continue;
                if ((widem >> c) & 1u)
                    far_chunk_fp32<IPL, true>(s_hi + h * TC, s_p + h * TC, xh, yh, zh, xr, yr, zr,
                                              ax, ay, az, ap);
                else
                    far_chunk_fp32<IPL, false>(s_hi + h * TC, s_p + h * TC, xh, yh, zh, xr, yr, zr,
                                               ax, ay, az, ap);
            }
        }
    }
    // the wave's deferred near chunks
    if (FUSED && nlist > 0) {
        double Hi[IPL], invHi[IPL], hi2[IPL];
        int idi[IPL];
        near_i_state<IPL>(I, ii, Hi, invHi, hi2, idi);
        wave_lds_sync();
        for (int q = 0; q < nlist; ++q) {
            const uint32_t e = s_near[wv].list[q];
            const int t = b.t0 + (int)(e >> 4) * b.tstep;
            for (int c = 0; c < CHUNKS; ++c)
                if ((e >> c) & 1u)
                    near_chunk_slice<IPL, NK>(s_near[wv], J, t, c, Ox, Oy, Oz, xr, yr, zr, Hi,
                                              invHi, hi2, idi, ax, ay, az, ap, nfp64);
        }
    }

#pragma unroll
    for (int k = 0; k < IPL; ++k) {
        if (!valid[k]) continue;
        b.part[ii[k]] = ax[k];
        b.part[b.pstride + ii[k]] = ay[k];
        b.part[2 * b.pstride + ii[k]] = az[k];
        b.part[3 * b.pstride + ii[k]] = ap[k];
    }
    if (stats) {
        // i past the end of the set (copies of the last one) are not counted
        unsigned f = 0;
#pragma unroll
        for (int k = 0; k < IPL; ++k) f += valid[k] ? nfp64[k] : 0u;
        const unsigned long long fw = wave_sum_count(f);
        if (lane == 0) {
            unsigned long long *st = stat_copy(stats);
            atomicAdd(&st[0], (unsigned long long)((b.t1 - b.t0 + b.tstep - 1) / b.tstep) * CHUNKS);
            atomicAdd(&st[1], (unsigned long long)nearv);
            atomicAdd(&st[2], (unsigned long long)widev);
            atomicAdd(&st[3], fw);
        }
    }
}

// ------------------------------------------------------- far block, FP64
template <int WG, int IPL>
__device__ __forceinline__ void far_block_fp64(const SortedSet &I, const SortedSet &J,
                                               const TileMeta *tiles, const TileMeta *chunks,
                                               const Block &b, unsigned long long *stats,
                                               double4 *s_p)
{
    constexpr int WI = 64 * IPL;
    constexpr int GI = WG * IPL;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;

    const int64_t io = min(b.ibase + GI / 2, b.iend - 1);
    const double Ox = I.x[io], Oy = I.y[io], Oz = I.z[io];

    double xr[IPL], yr[IPL], zr[IPL];
    float xf[IPL], yf[IPL], zf[IPL], hf[IPL];
    int64_t ii[IPL];
    bool valid[IPL];
    float bl[3] = {INFINITY, INFINITY, INFINITY}, bh[3] = {-INFINITY, -INFINITY, -INFINITY};
    float hmax = 0.0f;
#pragma unroll
    for (int k = 0; k < IPL; ++k) {
        const int64_t i = b.ibase + wv * WI + k * 64 + lane;
        valid[k] = i < b.iend;
        ii[k] = valid[k] ? i : b.iend - 1;
        xr[k] = I.x[ii[k]] - Ox;
        yr[k] = I.y[ii[k]] - Oy;
        zr[k] = I.z[ii[k]] - Oz;
        // the same FP32 positions as the FP32 kernel, so both classify tiles alike
        xf[k] = (float)xr[k];
        yf[k] = (float)yr[k];
        zf[k] = (float)zr[k];
        hf[k] = (float)fabs(I.Hs[ii[k]]);
        bl[0] = fminf(bl[0], xf[k]); bl[1] = fminf(bl[1], yf[k]); bl[2] = fminf(bl[2], zf[k]);
        bh[0] = fmaxf(bh[0], xf[k]); bh[1] = fmaxf(bh[1], yf[k]); bh[2] = fmaxf(bh[2], zf[k]);
        hmax = fmaxf(hmax, hf[k]);
    }
    for (int c = 0; c < 3; ++c) {
        bl[c] = wave_min(bl[c]);
        bh[c] = wave_max(bh[c]);
    }
    hmax = wave_max(hmax);

    double ax[IPL], ay[IPL], az[IPL], ap[IPL];
#pragma unroll
    for (int k = 0; k < IPL; ++k) ax[k] = ay[k] = az[k] = ap[k] = 0.0;

    const bool active = uniform_i(b.ibase + wv * WI < b.iend) != 0;
    unsigned nearv = 0;
    unsigned char *flags = b.flags + wv * b.fstride;
    for (int t = b.t0; t < b.t1; t += b.tstep) {
        const TileMeta &tm = tiles[t];
        const unsigned mask =
            active ? near_mask<IPL>(chunks, t, tm, box_dist2(tm, Ox, Oy, Oz, bl, bh), Ox, Oy, Oz,
                                    bl, bh, hmax, xf, yf, zf, hf)
                   : 0u;
        if (lane == 0) flags[t - b.fbase] = (unsigned char)mask;
        nearv += __builtin_popcount(mask);
        if (WG == 64 && mask == (1u << CHUNKS) - 1) continue;
        for (int s = 0; s < TJ / TS; ++s) {
            __syncthreads();
            for (int jj = tid; jj < TS; jj += WG) {
                const int64_t j = (int64_t)t * TJ + s * TS + jj;
                s_p[jj] = make_double4(J.x[j] - Ox, J.y[j] - Oy, J.z[j] - Oz, J.m[j]);
            }
            __syncthreads();
            if (!active) continue;
            for (int h = 0; h < TS / TC; ++h) {
                if ((mask >> (s * (TS / TC) + h)) & 1u) continue;
#pragma unroll 2
                for (int jj = h * TC; jj < (h + 1) * TC; ++jj) {
                    const double4 q = s_p[jj];
#pragma unroll
                    for (int k = 0; k < IPL; ++k) {
                        const double dx = q.x - xr[k], dy = q.y - yr[k], dz = q.z - zr[k];
                        const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
                        const double ri = rsqrt_pos64(r2);   // far: r^2 >= max(H_i^2, H_j^2) > 0
                        const double mr = q.w * ri;
                        const double mr3 = mr * ri * ri;
                        ax[k] = fma(mr3, dx, ax[k]);
                        ay[k] = fma(mr3, dy, ay[k]);
                        az[k] = fma(mr3, dz, az[k]);
                        ap[k] -= mr;
                    }
                }
            }
        }
    }

#pragma unroll
    for (int k = 0; k < IPL; ++k) {
        if (!valid[k]) continue;
        b.part[ii[k]] = ax[k];
        b.part[b.pstride + ii[k]] = ay[k];
        b.part[2 * b.pstride + ii[k]] = az[k];
        b.part[3 * b.pstride + ii[k]] = ap[k];
    }
    if (stats && lane == 0) {
        unsigned long long *st = stat_copy(stats);
        atomicAdd(&st[0], (unsigned long long)((b.t1 - b.t0 + b.tstep - 1) / b.tstep) * CHUNKS);
        atomicAdd(&st[1], (unsigned long long)nearv);
    }
}

// ------------------------------------------------------------ near group
// One workgroup of NEAR_WAVES waves per i-group.  The waves deal the group's
// flagged tiles round-robin among themselves, stage each tile in 64-particle
// chunks in their own LDS slice, and at the end combine their sums in a
// fixed order (wave 0 + 1 + 2 + 3) before adding them to the far kernel's
// partials.
__device__ __forceinline__ bool group_has_near(const Group &g)
{
    for (int t = g.t0; t < g.t1; ++t)
        if (g.flags[t - g.t0]) return true;
    return false;
}

constexpr int NEAR_CHUNK = TC;   // j per LDS chunk of a near wave (one per lane)
static_assert(NEAR_CHUNK == 64, "one staged particle per lane");

// 18 KB per workgroup, so LDS does not cap occupancy below the register limit
struct NearLds {
    double4 p[NEAR_WAVES][NEAR_CHUNK];   // x, y, z relative to the origin; m
    double4 h[NEAR_WAVES][NEAR_CHUNK];   // signed H, original index (as double), 1/|H|, H^2
    float2 mh[NEAR_WAVES][NEAR_CHUNK];   // FP32 m, H^2 (FAST kernels)
};

// With PSI (IPL = 1 only) it also forms the grad-h softening term
// psi_i = -(2/H_i^2) sum_j m_j (P(q_i) + q_i^2 A(q_i)) of gas particles i and
// adds it to g.psipart.
template <int IPL, bool FAST, int NK, bool PSI = false>
__device__ __forceinline__ void near_group(const SortedSet &I, const SortedSet &J,
                                           const Group &g, NearLds &lds, double *s_red)
{
    static_assert(!PSI || IPL == 1, "psi is formed with one i per lane");
    constexpr int NC = PSI ? 5 : 4;   // sums per i: ax, ay, az, pot (, psi)
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int64_t io = min(g.gbase + 32 * IPL, g.iend - 1);
    const double Ox = I.x[io], Oy = I.y[io], Oz = I.z[io];

    double xr[IPL], yr[IPL], zr[IPL], Hi[IPL], invHi[IPL], hi2[IPL];
    double ax[IPL], ay[IPL], az[IPL], ap[IPL], ps[IPL];
    int idi[IPL];
    int64_t ii[IPL];
    bool valid[IPL];
#pragma unroll
    for (int k = 0; k < IPL; ++k) {
        const int64_t i = g.gbase + k * 64 + lane;
        valid[k] = i < g.iend;
        ii[k] = valid[k] ? i : g.iend - 1;
        xr[k] = I.x[ii[k]] - Ox;
        yr[k] = I.y[ii[k]] - Oy;
        zr[k] = I.z[ii[k]] - Oz;
        Hi[k] = fabs(I.Hs[ii[k]]);
        invHi[k] = 1.0 / Hi[k];
        hi2[k] = Hi[k] * Hi[k];
        idi[k] = I.idx[ii[k]];
        ax[k] = ay[k] = az[k] = ap[k] = ps[k] = 0.0;
    }

    // FP32 H_i^2 for the FAST kernels' softened-pair test
    float hi2f[IPL];
#pragma unroll
    for (int k = 0; k < IPL; ++k) hi2f[k] = (float)hi2[k];

    int cnt = 0;
    for (int t = g.t0; t < g.t1; ++t) {
        const unsigned fl = g.flags[t - g.t0];
        if (!fl) continue;
        if ((cnt++ % NEAR_WAVES) != w) continue;
        for (int c0 = 0; c0 < TJ; c0 += NEAR_CHUNK) {
            if (!((fl >> (c0 / TC)) & 1u)) continue;   // a far chunk of a near tile
            const int64_t j = (int64_t)t * TJ + c0 + lane;
            wave_lds_sync();
            const double jx = J.x[j] - Ox, jy = J.y[j] - Oy, jz = J.z[j] - Oz;
            lds.p[w][lane] = make_double4(jx, jy, jz, J.m[j]);
            const double hs = J.Hs[j], ha = fabs(hs);
            lds.h[w][lane] = make_double4(hs, (double)J.idx[j], 1.0 / ha, ha * ha);
            if (FAST) lds.mh[w][lane] = make_float2((float)J.m[j], (float)(ha * ha));
            wave_lds_sync();
            if (FAST) {
                // Newtonian pairs in FP32 (differences formed in FP64 and
                // rounded once, as in the forward near tail; sums folded into
                // FP64 every FOLD j); the pairs with r^2 < max(H_i^2, H_j^2),
                // including r = 0, go on their lane's list and then take the
                // FP64 pair, each lane walking its own list.
                uint64_t own[IPL];
#pragma unroll
                for (int k = 0; k < IPL; ++k) own[k] = 0;
                for (int f0 = 0; f0 < NEAR_CHUNK; f0 += FOLD) {
                    float fx[IPL], fy[IPL], fz[IPL], fp[IPL];
#pragma unroll
                    for (int k = 0; k < IPL; ++k) fx[k] = fy[k] = fz[k] = fp[k] = 0.0f;
#pragma unroll 2
                    for (int jj = f0; jj < f0 + FOLD; ++jj) {
                        const double4 pd = lds.p[w][jj];
                        const float2 mh = lds.mh[w][jj];   // m_j, H_j^2
#pragma unroll
                        for (int k = 0; k < IPL; ++k) {
                            const float dx = (float)(pd.x - xr[k]);
                            const float dy = (float)(pd.y - yr[k]);
                            const float dz = (float)(pd.z - zr[k]);
                            const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                            const bool soft = r2 < fmaxf(hi2f[k], mh.y);
                            const float ri = soft ? 0.0f : __builtin_amdgcn_rsqf(r2);
                            const float mr = mh.x * ri;
                            const float mr3 = mr * ri * ri;
                            fx[k] = fmaf(mr3, dx, fx[k]);
                            fy[k] = fmaf(mr3, dy, fy[k]);
                            fz[k] = fmaf(mr3, dz, fz[k]);
                            fp[k] += mr;
                            if (soft) own[k] |= 1ull << jj;
                        }
                    }
#pragma unroll
                    for (int k = 0; k < IPL; ++k) {
                        ax[k] += (double)fx[k];
                        ay[k] += (double)fy[k];
                        az[k] += (double)fz[k];
                        ap[k] -= (double)fp[k];
                    }
                }
#pragma unroll
                for (int k = 0; k < IPL; ++k) {
                    while (own[k]) {
                        const int jj = __builtin_ctzll(own[k]);
                        own[k] &= own[k] - 1;
                        const double4 p = lds.p[w][jj];
                        const double4 h = lds.h[w][jj];
                        near_pair<FAST, NK, PSI>(p.x - xr[k], p.y - yr[k], p.z - zr[k], Hi[k],
                                                 invHi[k], hi2[k], fabs(h.x), h.z, h.w, p.w,
                                                 h.x > 0.0, (int)h.y == idi[k], ax[k], ay[k],
                                                 az[k], ap[k], &ps[k]);
                    }
                }
            } else {
#pragma unroll 1
                for (int jj = 0; jj < NEAR_CHUNK; ++jj) {
                    const double4 p = lds.p[w][jj];
                    const double4 h = lds.h[w][jj];
#pragma unroll
                    for (int k = 0; k < IPL; ++k)
                        near_pair<FAST, NK, PSI>(p.x - xr[k], p.y - yr[k], p.z - zr[k], Hi[k],
                                                 invHi[k], hi2[k], fabs(h.x), h.z, h.w, p.w,
                                                 h.x > 0.0, (int)h.y == idi[k], ax[k], ay[k],
                                                 az[k], ap[k], &ps[k]);
                }
            }
        }
    }

    // fixed-order combination of the waves' sums, added to the partials
    if (w > 0) {
#pragma unroll
        for (int k = 0; k < IPL; ++k) {
            double *r = s_red + (((w - 1) * NC) * IPL + k) * 64 + lane;
            r[0] = ax[k];
            r[IPL * 64] = ay[k];
            r[2 * IPL * 64] = az[k];
            r[3 * IPL * 64] = ap[k];
            if (PSI) r[4 * IPL * 64] = ps[k];
        }
    }
    __syncthreads();
    if (w != 0) return;
#pragma unroll
    for (int k = 0; k < IPL; ++k) {
        for (int v = 0; v < NEAR_WAVES - 1; ++v) {
            const double *r = s_red + ((v * NC) * IPL + k) * 64 + lane;
            ax[k] += r[0];
            ay[k] += r[IPL * 64];
            az[k] += r[2 * IPL * 64];
            ap[k] += r[3 * IPL * 64];
            if (PSI) ps[k] += r[4 * IPL * 64];
        }
        if (!valid[k]) continue;
        g.part[ii[k]] += ax[k];
        g.part[g.pstride + ii[k]] += ay[k];
        g.part[2 * g.pstride + ii[k]] += az[k];
        g.part[3 * g.pstride + ii[k]] += ap[k];
        // point particles (negative H) carry no psi (advance.f90:750-753)
        if (PSI && I.Hs[ii[k]] > 0.0)
            g.psipart[ii[k]] += -2.0 * invHi[k] * invHi[k] * ps[k];
    }
}

// ======================================================= single-set kernels
__device__ __forceinline__ void tile_range(const PairArgs &a, int jp, int &t0, int &t1)
{
    t0 = (int)((int64_t)a.ntiles * jp / a.jsplit);
    t1 = (int)((int64_t)a.ntiles * (jp + 1) / a.jsplit);
}

template <int WG, int IPL>
__device__ __forceinline__ Block single_block(const PairArgs &a)
{
    const int ib = blockIdx.x % a.niblocks;
    const int jp = blockIdx.x / a.niblocks;
    Block b;
    b.ibase = (int64_t)ib * WG * IPL;
    b.iend = a.ni;
    // partition jp takes every jsplit-th tile: the near tiles of a wave,
    // neighbours along the curve, spread over the partitions instead of
    // piling up in one
    b.t0 = jp;
    b.t1 = a.ntiles;
    b.tstep = a.jsplit;
    b.fbase = 0;
    b.fstride = a.ntiles;
    b.flags = a.nearflag + (int64_t)ib * (WG / 64) * a.ntiles;
    b.part = a.partial + (int64_t)jp * 4 * a.ni;
    b.pstride = a.ni;
    return b;
}

// The forward FP32C pass: far and near chunks in one kernel.  With one i per
// lane the register budget is held to 7 waves per SIMD, the occupancy of the
// far loop alone; the near chunks' FP64 fallback then spills a few values
// to scratch outside the pair loops.
template <int WG, int IPL, int NK>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(IPL == 1 ? 7 : 1)))
void k_far_fp32c(PairArgs a)
{
    __shared__ float4 s_hi[TS];
    __shared__ double4 s_p[TS];
    __shared__ NearSlice s_near[WG / 64];
    far_block_fp32c<WG, IPL, NK, true>(a.i, a.j, a.tiles, a.chunks, single_block<WG, IPL>(a),
                                       a.stats, s_hi, s_p, s_near);
}

// Far chunks only, near chunks flagged (the pass with the grad-h term).
template <int WG>
__global__ __launch_bounds__(WG) void k_far_fp32c_split(PairArgs a)
{
    __shared__ float4 s_hi[TS];
    __shared__ double4 s_p[TS];
    far_block_fp32c<WG, 1, 0, false>(a.i, a.j, a.tiles, a.chunks, single_block<WG, 1>(a),
                                     a.stats, s_hi, s_p, nullptr);
}

template <int WG, int IPL>
__global__ __launch_bounds__(WG) void k_far_fp64(PairArgs a)
{
    __shared__ double4 s_p[TS];
    far_block_fp64<WG, IPL>(a.i, a.j, a.tiles, a.chunks, single_block<WG, IPL>(a), a.stats, s_p);
}

template <int IPL, bool FAST, int NK>
__global__ __launch_bounds__(64 * NEAR_WAVES) void k_near(PairArgs a)
{
    __shared__ NearLds lds;
    __shared__ double s_red[(NEAR_WAVES - 1) * 4 * IPL * 64];
    const int64_t gi = blockIdx.x % a.ngroups;
    const int jp = (int)(blockIdx.x / a.ngroups);
    Group g;
    g.gbase = gi * (64 * IPL);
    g.iend = a.ni;
    tile_range(a, jp, g.t0, g.t1);
    g.flags = a.nearflag + gi * a.ntiles + g.t0;
    g.part = a.partial + (int64_t)jp * 4 * a.ni;
    g.pstride = a.ni;
    if (g.gbase >= g.iend || !group_has_near(g)) return;
    near_group<IPL, FAST, NK>(a.i, a.j, g, lds, s_red);
}

// Near kernel that also forms the grad-h softening term (one i per lane).
template <bool FAST, int NK>
__global__ __launch_bounds__(64 * NEAR_WAVES) void k_near_psi(PairArgs a)
{
    __shared__ NearLds lds;
    __shared__ double s_red[(NEAR_WAVES - 1) * 5 * 64];
    const int64_t gi = blockIdx.x % a.ngroups;
    const int jp = (int)(blockIdx.x / a.ngroups);
    Group g;
    g.gbase = gi * 64;
    g.iend = a.ni;
    tile_range(a, jp, g.t0, g.t1);
    g.flags = a.nearflag + gi * a.ntiles + g.t0;
    g.part = a.partial + (int64_t)jp * 4 * a.ni;
    g.pstride = a.ni;
    g.psipart = a.psipart + (int64_t)jp * a.ni;
    if (g.gbase >= g.iend || !group_has_near(g)) return;
    near_group<1, FAST, NK, true>(a.i, a.j, g, lds, s_red);
}

// ------------------------------------------------- one wave, one column chunk
// The kernels below evaluate chunk visits wave by wave: 64 i, one per lane,
// against the 64 j staged in the wave's slice.  Their pair loops run in
// groups of PG pairs whose v_rsq_f32 are issued together at raised wave
// priority: a v_rsq_f32 issues alone, and at equal priority the wave that is
// first past its own runs ahead and the two waves of a SIMD no longer issue
// their other FP32 instructions together (sg_sym.hip).
constexpr int PG = 4;

// LDS of a wave: the staged chunk, and the softened pairs of a visit dealt
// evenly over the lanes.
constexpr int NSOFT = 1024;   // listed pairs: a quarter of a visit's (visit_soft)
struct WaveLds {
    NearSlice sl;
    uint16_t list[NSOFT];     // i lane << 6 | j
    double res[5][64];        // sums of one pair per lane (ax, ay, az, pot, psi)
};

__device__ __forceinline__ void rsq_group(const float (&r2)[PG], float (&ri)[PG])
{
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(3);
#pragma unroll
    for (int u = 0; u < PG; ++u) ri[u] = __builtin_amdgcn_rsqf(r2[u]);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
}

// FP32 sums of one fold.
struct Fold4 {
    float x = 0.0f, y = 0.0f, z = 0.0f, p = 0.0f;
    __device__ __forceinline__ void add(float ri, float m, float dx, float dy, float dz)
    {
        const float mr = m * ri, mr3 = mr * ri * ri;
        x = fmaf(mr3, dx, x);
        y = fmaf(mr3, dy, y);
        z = fmaf(mr3, dz, z);
        p += mr;
    }
    template <int N>
    __device__ __forceinline__ void to(double (&acc)[N]) const
    {
        acc[0] += (double)x;
        acc[1] += (double)y;
        acc[2] += (double)z;
        acc[3] -= (double)p;
    }
};

enum Visit { VISIT_FAR, VISIT_WIDE, VISIT_NEAR };

// How the chunk with box and largest H cm is evaluated by a wave with one
// particle per lane at (px, py, pz) relative to O (distance^2 rho2 from it),
// support ph and box_slack slack: near when some lane's pairs may be softened, else wide when
// a lane is too close, relative to its distance from O, for differences of
// positions rounded relative to O.
__device__ __forceinline__ Visit classify_visit(const TileMeta &cm, double Ox, double Oy, double Oz,
                                                float px, float py, float pz, float ph, float slack,
                                                float rho2)
{
    const float gx = fmaxf(0.0f, fmaxf((float)(cm.lo[0] - Ox) - px, px - (float)(cm.hi[0] - Ox)));
    const float gy = fmaxf(0.0f, fmaxf((float)(cm.lo[1] - Oy) - py, py - (float)(cm.hi[1] - Oy)));
    const float gz = fmaxf(0.0f, fmaxf((float)(cm.lo[2] - Oz) - pz, pz - (float)(cm.hi[2] - Oz)));
    const float d2 = fmaf(gx, gx, fmaf(gy, gy, gz * gz));
    const float hm = fmaxf(ph, (float)cm.maxH) + slack;
    if (__ballot(!(d2 > hm * hm * (1.0f + FAR_MARGIN)))) return VISIT_NEAR;
    if (__ballot(!(d2 > WIDE_K * WIDE_K * rho2 * (1.0f + FAR_MARGIN)))) return VISIT_WIDE;
    return VISIT_FAR;
}

// One side of a softened pair without a branch: the polynomials, or the
// Newtonian terms beyond H.  q = 0 (r = 0, with ri passed as 0) gives the
// r -> 0 limit.
template <int NK>
__device__ __forceinline__ void side_select(double r, double ri, double r2, double H, double invH,
                                            double &gacc, double &gpot, double *ps = nullptr)
{
    const double q = r * invH;
    double A, P;
    if (NK == 0) cubic_AP(q, H * ri, A, P);
    else poly_AP(NK, q, 0.0, A, P);
    const bool soft = r2 <= H * H;
    gacc += soft ? A * invH * invH * invH : ri * ri * ri;
    gpot += soft ? P * invH : -ri;
    if (ps) *ps = soft ? fma(q * q, A, P) : 0.0;
}

// near_pair for a pair that is (or within rounding of being) softened, with
// no branch: dealt over the lanes such pairs take different ones, and a wave
// would walk them all.  dead: the self pair of a point particle.  With PSI
// f[4] is m_j (P(q_i) + q_i^2 A(q_i)) where r <= H_i, as in near_pair.
template <int NK, bool PSI, bool FAST>
__device__ __forceinline__ void soft_pair(double dx, double dy, double dz, double Hi, double invHi,
                                          double Hj, double invHj, double mj, bool dead,
                                          double (&f)[PSI ? 5 : 4])
{
    const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
    const bool apart = r2 > 0.0;
    const double ri = apart ? rsqrt64<FAST>(apart ? r2 : 1.0) : 0.0;
    const double r = r2 * ri;
    double gacc = 0.0, gpot = 0.0, ps = 0.0;
    side_select<NK>(r, ri, r2, Hi, invHi, gacc, gpot, PSI ? &ps : nullptr);
    side_select<NK>(r, ri, r2, Hj, invHj, gacc, gpot);
    const double hm = dead ? 0.0 : 0.5 * mj;
    const double g = hm * gacc;
    f[0] = g * dx;
    f[1] = g * dy;
    f[2] = g * dz;
    f[3] = hm * gpot;
    if (PSI) f[PSI ? 4 : 0] = mj * ps;
}

// The pairs that visit_near and visit64 leave: bit 63 - jj of `mine` is the
// lane's softened pair with jj of the staged chunk.  A lane has few of them and
// the busiest several times the mean, and one costs some 300 dependent FP64
// operations, so they are dealt over all lanes, 64 at a time, and each lane
// collects the sums of its own.  A quarter of the visit's `npairs` pairs is dealt at
// most: beyond it the busiest lane is near the mean and every lane walks its own
// (4,096 particles with supports three times the usual, visits of 16 columns: 0.31
// -> 0.15 ms).  DENSE, for FP64: `dense` tells whether more than half were
// softened; the next near visit then lists all its pairs, without the body for the
// others, a quarter of a softened pair's time.  65,537 particles with supports of
// ten and a hundred times the usual: 19.0 -> 14.6 and 19.8 -> 13.9 ms (tile kernels
// 12.9 and 13.7).  In FP32C that body costs as little as looking out for such
// visits.  Returns the lane's softened pairs, of particles.
template <int NK, bool PSI, bool FAST, bool DENSE>
__device__ __forceinline__ unsigned visit_soft(WaveLds &lds, uint64_t mine, uint64_t real,
                                               const SortedSet &J, int64_t j0c, double xr, double yr,
                                               double zr, double Hi, double invHi, double hi2, int idi,
                                               double (&acc)[PSI ? 5 : 4], unsigned npairs, bool &dense)
{
    constexpr int NS = PSI ? 5 : 4;
    const NearSlice &sl = lds.sl;
    const unsigned count = (unsigned)__builtin_popcountll(mine);
    unsigned at, total;
    list_places(count, at, total);
    // softened pairs with particles, not padding
    unsigned soft = (unsigned)__builtin_popcountll(mine & __brevll(real));
    if (4 * total > npairs) {
        if (DENSE) soft = 0;
        while (mine) {
            const int jj = __builtin_clzll(mine);
            mine &= ~(0x8000000000000000ull >> jj);
            const double4 p = sl.p[jj];
            const double hs = sl.hs[jj], Hj = fabs(hs), invHj = sl.hinv[jj], hj2 = Hj * Hj;
            const double dx = p.x - xr, dy = p.y - yr, dz = p.z - zr;
            // the self pair only matters at r = 0: the index is read then
            const bool same = dx == 0.0 && dy == 0.0 && dz == 0.0 && J.idx[j0c + jj] == idi;
            if (DENSE) {
                near_pair<FAST, NK, PSI>(dx, dy, dz, Hi, invHi, hi2, Hj, invHj, hj2, sl.m[jj], hs > 0.0,
                                         same, acc[0], acc[1], acc[2], acc[3], &acc[PSI ? 4 : 3]);
                if (fma(dx, dx, fma(dy, dy, dz * dz)) < fmax(hi2, hj2))
                    soft += (unsigned)(real >> jj & 1);
            } else {
                double f[NS];
                soft_pair<NK, PSI, FAST>(dx, dy, dz, Hi, invHi, Hj, invHj, sl.m[jj], same && hs < 0.0, f);
#pragma unroll
                for (int k = 0; k < NS; ++k) acc[k] += f[k];
            }
        }
        if (DENSE) {
            list_places(soft, at, total);
            dense = 2 * total > npairs;
        }
        return soft;
    }
    dense = false;
    const int lane = threadIdx.x & 63;
    for (unsigned k = at; mine; ++k) {
        const int jj = __builtin_clzll(mine);
        mine &= ~(0x8000000000000000ull >> jj);
        lds.list[k] = (uint16_t)(lane << 6 | jj);
    }
    for (unsigned b0 = 0; b0 < total; b0 += 64) {
        wave_lds_sync();
        const unsigned e = min(b0 + (unsigned)lane, total - 1);   // lanes past the end repeat the last
        const int il = lds.list[e] >> 6, jj = lds.list[e] & 63;
        const double4 p = sl.p[jj];
        const double hs = sl.hs[jj];
        const double H = __shfl(Hi, il, 64), invH = __shfl(invHi, il, 64);
        const int id = __shfl(idi, il, 64);
        const double dx = p.x - __shfl(xr, il, 64), dy = p.y - __shfl(yr, il, 64),
                     dz = p.z - __shfl(zr, il, 64);
        const bool dead = dx == 0.0 && dy == 0.0 && dz == 0.0 && hs < 0.0 && J.idx[j0c + jj] == id;
        double f[NS];
        soft_pair<NK, PSI, FAST>(dx, dy, dz, H, invH, fabs(hs), sl.hinv[jj], sl.m[jj], dead, f);
#pragma unroll
        for (int k = 0; k < NS; ++k) lds.res[k][lane] = f[k];
        wave_lds_sync();
        // each lane adds its own pairs, in the list's order
        const unsigned hi = min(at + count, b0 + 64);
        for (unsigned k = max(at, b0); k < hi; ++k) {
#pragma unroll
            for (int c = 0; c < NS; ++c) acc[c] += lds.res[c][k - b0];
        }
    }
    return soft;
}

// The visits below cover j = jb .. je - 1 of the staged chunk (multiples of
// PG).  Near: differences formed in FP64 and rounded once, the FP32 body for every
// pair (r^-1 = 0 for those that may be softened, r^2 < max(H_i^2, H_j^2) in
// FP32, r = 0 included), and those in FP64 (visit_soft).  PSI also forms the
// grad-h sum (acc[4]).
template <int NK, bool PSI>
__device__ __forceinline__ void visit_near(WaveLds &lds, uint64_t real, const SortedSet &J,
                                           int64_t j0c, int jb, int je, double xr, double yr, double zr, double Hi,
                                           double invHi, double hi2, int idi,
                                           double (&acc)[PSI ? 5 : 4],
                                           unsigned &nfp64)
{
    const NearSlice &sl = lds.sl;
    const float hi2f = (float)hi2;
    uint64_t mine = 0;   // bit 63 - jj: the lane's pair with jj is softened
#pragma unroll 1
    for (int f = jb; f < je; f += FOLD) {
        const int fe = min(f + FOLD, je);
        Fold4 sum;
        uint32_t list = 0;
#pragma unroll 1
        for (int j0 = f; j0 < fe; j0 += PG) {
            float dx[PG], dy[PG], dz[PG], m[PG], r2[PG], ri[PG];
#pragma unroll
            for (int u = 0; u < PG; ++u) {
                const double4 p = sl.p[j0 + u];
                const float2 mh = __builtin_bit_cast(float2, p.w);   // m_j, H_j^2
                dx[u] = (float)(p.x - xr);
                dy[u] = (float)(p.y - yr);
                dz[u] = (float)(p.z - zr);
                m[u] = mh.x;
                const float q = fmaf(dx[u], dx[u], fmaf(dy[u], dy[u], dz[u] * dz[u]));
                const bool soft = q < fmaxf(hi2f, mh.y);
                r2[u] = soft ? INFINITY : q;
                list = list + list + (soft ? 1u : 0u);
            }
            rsq_group(r2, ri);
#pragma unroll
            for (int u = 0; u < PG; ++u) sum.add(ri[u], m[u], dx[u], dy[u], dz[u]);
        }
        sum.to(acc);
        mine |= (uint64_t)list << (TC - fe);
    }
    bool dense = false;
    nfp64 += visit_soft<NK, PSI, true, false>(lds, mine, real, J, j0c, xr, yr, zr, Hi, invHi, hi2, idi,
                                              acc, 64 * (je - jb), dense);
}

// Near and far chunks of an FP64 pass.
template <int NK, bool NEAR, bool PSI>
__device__ __forceinline__ void visit64(WaveLds &lds, uint64_t real, const SortedSet &J, int64_t j0c,
                                        double xr, double yr, double zr, double Hi, double invHi,
                                        double hi2, int idi, double (&acc)[PSI ? 5 : 4], bool &dense)
{
    const NearSlice &sl = lds.sl;
    uint64_t mine = NEAR && dense ? ~0ull : 0;
#pragma unroll 4
    for (int j = NEAR && dense ? TC : 0; j < TC; ++j) {
        const double4 p = sl.p[j];
        const double dx = p.x - xr, dy = p.y - yr, dz = p.z - zr;
        double r2 = fma(dx, dx, fma(dy, dy, dz * dz)), m = sl.m[j];
        if (NEAR) {
            const bool soft = r2 < fmax(hi2, sl.hs[j] * sl.hs[j]);
            r2 = soft ? 1.0 : r2;
            m = soft ? 0.0 : m;
            mine = mine + mine + (soft ? 1u : 0u);
        }
        const double ri = rsqrt_pos64(r2);
        const double mr = m * ri, mr3 = mr * ri * ri;
        acc[0] = fma(mr3, dx, acc[0]);
        acc[1] = fma(mr3, dy, acc[1]);
        acc[2] = fma(mr3, dz, acc[2]);
        acc[3] -= mr;
    }
    if (NEAR)
        visit_soft<NK, PSI, false, true>(lds, mine, real, J, j0c, xr, yr, zr, Hi, invHi, hi2, idi, acc,
                                         64 * TC, dense);
}

// Wide: as near, with every pair Newtonian.
template <int N>
__device__ __forceinline__ void visit_wide(const NearSlice &sl, int jb, int je, double xr, double yr,
                                           double zr, double (&acc)[N])
{
#pragma unroll 1
    for (int f = jb; f < je; f += FOLD) {
        const int fe = min(f + FOLD, je);
        Fold4 sum;
#pragma unroll 2
        for (int j0 = f; j0 < fe; j0 += PG) {
            float dx[PG], dy[PG], dz[PG], m[PG], r2[PG], ri[PG];
#pragma unroll
            for (int u = 0; u < PG; ++u) {
                const double4 p = sl.p[j0 + u];
                dx[u] = (float)(p.x - xr);
                dy[u] = (float)(p.y - yr);
                dz[u] = (float)(p.z - zr);
                m[u] = __builtin_bit_cast(float2, p.w).x;
                r2[u] = fmaf(dx[u], dx[u], fmaf(dy[u], dy[u], dz[u] * dz[u]));
            }
            rsq_group(r2, ri);
#pragma unroll
            for (int u = 0; u < PG; ++u) sum.add(ri[u], m[u], dx[u], dy[u], dz[u]);
        }
        sum.to(acc);
    }
}

// Far: differences of FP32 positions relative to O.
template <int N>
__device__ __forceinline__ void visit_far(const float4 *s_hi, int jb, int je, float xh, float yh,
                                          float zh, double (&acc)[N])
{
#pragma unroll 1
    for (int f = jb; f < je; f += FOLD) {
        const int fe = min(f + FOLD, je);
        Fold4 sum;
#pragma unroll 2
        for (int j0 = f; j0 < fe; j0 += PG) {
            float dx[PG], dy[PG], dz[PG], m[PG], r2[PG], ri[PG];
#pragma unroll
            for (int u = 0; u < PG; ++u) {
                const float4 p = s_hi[j0 + u];
                dx[u] = p.x - xh;
                dy[u] = p.y - yh;
                dz[u] = p.z - zh;
                m[u] = p.w;
                r2[u] = fmaf(dx[u], dx[u], fmaf(dy[u], dy[u], dz[u] * dz[u]));
            }
            rsq_group(r2, ri);
#pragma unroll
            for (int u = 0; u < PG; ++u) sum.add(ri[u], m[u], dx[u], dy[u], dz[u]);
        }
        sum.to(acc);
    }
}

// ------------------------------------------------------ wave-sized work items
// The forward FP32C pass of small i-ranges: one wave per 64 i and j partition
// (strided chunks, or parts of them), so that a few thousand particles still
// make thousands of waves and a wave's near chunks are few.  The next chunk's
// particles are loaded while the current one is evaluated.
template <int NK, bool PSI>
__global__ __launch_bounds__(64) void k_pair_wave(PairArgs a)
{
    __shared__ WaveLds lds;
    NearSlice &sl = lds.sl;
    const int lane = threadIdx.x;
    const unsigned nic = (unsigned)((a.ni + TC - 1) / TC);
    const int ci = (int)(blockIdx.x % nic), jp = (int)(blockIdx.x / nic);
    const int nchunks = a.ntiles * CHUNKS;
    const int64_t gbase = (int64_t)ci * TC;
    const int64_t io = min(gbase + TC / 2, a.ni - 1);
    const double Ox = a.i.x[io], Oy = a.i.y[io], Oz = a.i.z[io];
    const bool valid = gbase + lane < a.ni;
    const int64_t ii[1] = {valid ? gbase + lane : a.ni - 1};
    const double xr = a.i.x[ii[0]] - Ox, yr = a.i.y[ii[0]] - Oy, zr = a.i.z[ii[0]] - Oz;
    double Hi[1], invHi[1], hi2[1];
    int idi[1];
    near_i_state<1>(a.i, ii, Hi, invHi, hi2, idi);
    const float px = (float)xr, py = (float)yr, pz = (float)zr, ph = (float)Hi[0];
    const float rho2 = fmaf(px, px, fmaf(py, py, pz * pz)), slack = box_slack(px, py, pz);
    double acc[PSI ? 5 : 4] = {};
    unsigned nfp64 = 0, visits = 0, nearv = 0, widev = 0;
    // partition jp: part jp % jsub of every (jsplit / jsub)-th chunk
    const int stride = a.jsplit / a.jsub, first = jp / a.jsub;
    const int jb = jp % a.jsub * (TC / a.jsub), je = jb + TC / a.jsub;
    int64_t j = (int64_t)first * TC + lane;
    double jx = a.j.x[j], jy = a.j.y[j], jz = a.j.z[j], jm = a.j.m[j], jh = a.j.Hs[j];
    for (int cj = first; cj < nchunks; cj += stride) {
        const Visit v = classify_visit(a.chunks[cj], Ox, Oy, Oz, px, py, pz, ph, slack, rho2);
        const double rx = jx - Ox, ry = jy - Oy, rz = jz - Oz;
        uint64_t real = 0;
        if (v == VISIT_FAR) {
            wave_lds_sync();
            reinterpret_cast<float4 *>(sl.p)[lane] =
                make_float4((float)rx, (float)ry, (float)rz, (float)jm);
            wave_lds_sync();
        } else {
            real = near_stage(sl, rx, ry, rz, jm, jh);
        }
        const int64_t j0c = (int64_t)cj * TC;
        if (cj + stride < nchunks) {
            j = j0c + (int64_t)stride * TC + lane;
            jx = a.j.x[j];
            jy = a.j.y[j];
            jz = a.j.z[j];
            jm = a.j.m[j];
            jh = a.j.Hs[j];
        }
        ++visits;
        if (v == VISIT_NEAR) {
            ++nearv;
            visit_near<NK, PSI>(lds, real, a.j, j0c, jb, je, xr, yr, zr, Hi[0], invHi[0], hi2[0], idi[0], acc, nfp64);
        } else if (v == VISIT_WIDE) {
            ++widev;
            visit_wide(sl, jb, je, xr, yr, zr, acc);
        } else {
            visit_far(reinterpret_cast<const float4 *>(sl.p), jb, je, px, py, pz, acc);
        }
    }
    if (valid) {
        double *part = a.partial + (int64_t)jp * 4 * a.ni + ii[0];
#pragma unroll
        for (int k = 0; k < 4; ++k) part[k * a.ni] = acc[k];
        // point particles (negative H) carry no psi (advance.f90:750-753)
        if (PSI)
            a.psipart[(int64_t)jp * a.ni + ii[0]] =
                a.i.Hs[ii[0]] > 0.0 ? -2.0 * invHi[0] * invHi[0] * acc[PSI ? 4 : 0] : 0.0;
    }
    if (a.stats) {
        const unsigned long long fw = wave_sum_count(valid ? nfp64 : 0u);
        if (lane == 0) {
            unsigned long long *st = stat_copy(a.stats);
            if (jb == 0) {   // a divided chunk is one visit
                atomicAdd(&st[0], (unsigned long long)visits);
                atomicAdd(&st[1], (unsigned long long)nearv);
                atomicAdd(&st[2], (unsigned long long)widev);
            }
            atomicAdd(&st[3], fw);
        }
    }
}

// ------------------------------------------- ordered rest of a whole-set pass
// The (row chunk, column chunk) visits that k_sym leaves (bits unset in
// a.sym): near chunks and those too close to the row chunk for hi-only
// differences.  One wave per segment of a row's visits, so that the rows that
// meet thousands of chunks (those of the largest H, and those that straddle a
// jump of the curve) do not outlast the rest.  The next chunk's particles are
// loaded while the current one is evaluated.
// With PSI it also forms the grad-h sums: all softened pairs are its own
// (forces and term, pair kernels, against the ordered pass with a near kernel:
// 50,000 particles 1.59 -> 1.34 ms, 65,536 2.23 -> 1.61, 131,072 6.26 -> 4.24).
template <int NK, bool FP64, bool PSI>
__global__ __launch_bounds__(64) void k_sym_rest(SymArgs a)
{
    __shared__ WaveLds lds;
    NearSlice &sl = lds.sl;
    const int lane = threadIdx.x;
    const int g = (int)blockIdx.x;
    if (g >= a.segtot[0]) return;
    int ci = segment_row(a.seg, a.nchunks, g);
    const int len = uniform_i(a.segtot[1]);
    const int k0 = uniform_i(g - a.seg[ci]) * len;
    if (a.sets) {
        const int set = a.setof[ci];
        ci -= uniform_i(a.sets[set].chunk0);
        a = sym_view(a, set);
    }
    const SortedSet &P = a.p;
    const int64_t gbase = (int64_t)ci * TC;
    const int64_t io = min(gbase + TC / 2, a.n - 1);
    const double Ox = P.x[io], Oy = P.y[io], Oz = P.z[io];
    const bool valid = gbase + lane < a.n;
    const int64_t ii[1] = {valid ? gbase + lane : a.n - 1};
    const double xr = P.x[ii[0]] - Ox, yr = P.y[ii[0]] - Oy, zr = P.z[ii[0]] - Oz;
    double Hi[1], invHi[1], hi2[1];
    int idi[1];
    near_i_state<1>(P, ii, Hi, invHi, hi2, idi);
    const float px = (float)xr, py = (float)yr, pz = (float)zr, ph = (float)Hi[0];
    const float rho2 = fmaf(px, px, fmaf(py, py, pz * pz)), slack = box_slack(px, py, pz);
    constexpr int NS = PSI ? 5 : 4;
    double acc[NS] = {};
    unsigned nfp64 = 0, visits = 0, nearv = 0, widev = 0;
    bool dense = false;   // of the last near visit

    RestBits it;
    it.row = a.sym + (int64_t)ci * a.words;
    it.nchunks = a.nchunks;
    it.words = a.words;
    // visits of this segment: a row's last one is the short one
    int left = min(len, rest_total(it.row, a.nchunks, a.words) - k0);
    it.start(k0);
    int cj = it.next();
    double jx = P.x[(int64_t)cj * TC + lane], jy = P.y[(int64_t)cj * TC + lane],
           jz = P.z[(int64_t)cj * TC + lane], jm = P.m[(int64_t)cj * TC + lane],
           jh = P.Hs[(int64_t)cj * TC + lane];
    for (;;) {
        const Visit v =
            classify_visit(a.chunks[cj], Ox, Oy, Oz, px, py, pz, ph, slack, FP64 ? 0.0f : rho2);
        const double rx = jx - Ox, ry = jy - Oy, rz = jz - Oz;
        uint64_t real = 0;
        if (!FP64 && v == VISIT_FAR) {
            wave_lds_sync();
            reinterpret_cast<float4 *>(sl.p)[lane] =
                make_float4((float)rx, (float)ry, (float)rz, (float)jm);
            wave_lds_sync();
        } else {
            real = near_stage(sl, rx, ry, rz, jm, jh);
        }
        const int64_t j0c = (int64_t)cj * TC;
        ++visits;
        if (--left > 0) {
            cj = it.next();
            const int64_t j = (int64_t)cj * TC + lane;
            jx = P.x[j];
            jy = P.y[j];
            jz = P.z[j];
            jm = P.m[j];
            jh = P.Hs[j];
        }
        if (v == VISIT_NEAR) ++nearv;
        if (FP64) {
            if (v == VISIT_NEAR)
                visit64<NK, true, PSI>(lds, real, P, j0c, xr, yr, zr, Hi[0], invHi[0], hi2[0], idi[0], acc, dense);
            else
                visit64<NK, false, PSI>(lds, real, P, j0c, xr, yr, zr, Hi[0], invHi[0], hi2[0], idi[0], acc, dense);
        } else if (v == VISIT_NEAR) {
            visit_near<NK, PSI>(lds, real, P, j0c, 0, TC, xr, yr, zr, Hi[0], invHi[0], hi2[0],
                                idi[0], acc, nfp64);
        } else if (v == VISIT_WIDE) {
            ++widev;
            visit_wide(sl, 0, TC, xr, yr, zr, acc);
        } else {
            visit_far(reinterpret_cast<const float4 *>(sl.p), 0, TC, px, py, pz, acc);
        }
        if (left <= 0) break;
    }
    double *s = a.segsum + (int64_t)g * NS * TC + lane;
#pragma unroll
    for (int k = 0; k < NS; ++k) s[k * TC] = acc[k];
    if (a.stats) {
        const unsigned long long fw = wave_sum_count(valid ? nfp64 : 0u);
        if (lane == 0) {
            unsigned long long *st = stat_copy(a.stats);
            atomicAdd(&st[0], (unsigned long long)visits);
            atomicAdd(&st[1], (unsigned long long)nearv);
            atomicAdd(&st[2], (unsigned long long)widev);
            atomicAdd(&st[3], fw);
        }
    }
}

// ------------------------------------------------- grad-h term on its own
// psi_i = -(2/H_i^2) sum_{j: r <= H_i} m_j (P(q_i) + q_i^2 A(q_i)) of the
// gas particles of the i-set, without the accelerations.  One wave per
// 64-particle i-group and part (every jsplit-th chunk): its lanes test 64 tiles
// at a time against the group's box (r <= H_i needs only the wave's largest H),
// then chunks, then each chunk against every lane's own reach.  The pairs of a
// chunk that may be within H_i (an FP32 test with a margin for its rounding)
// are listed and dealt over the lanes as in visit_soft, since a lane has about
// one in a chunk, and decided and evaluated in FP64.  What bounds it are the
// chunk tests of the groups whose box or largest H reaches most of the set, so
// the parts share the tests and not only the visits.  65,536 particles: kernel
// 0.50 ms with every part testing all chunks, whole call 0.88 -> 0.57 ms (0.80
// from the FP32 test alone); 200,000 2.47 -> 1.49 ms.
struct PsiLds {
    double4 p[TC];
    float4 f[TC];             // the positions rounded to FP32
    uint16_t list[NSOFT];
    double res[64];
};

template <int NK>
__device__ __forceinline__ double psi_pair(double dx, double dy, double dz, double H, double invH,
                                           double mj)
{
    const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
    if (r2 > H * H) return 0.0;   // listed by the FP32 test's margin
    const bool apart = r2 > 0.0;
    const double ri = apart ? rsqrt_pos64(apart ? r2 : 1.0) : 0.0;
    const double r = r2 * ri, q = r * invH;
    double A, P;
    if (NK == 0) cubic_AP(q, H * ri, A, P);
    else poly_AP(NK, q, 0.0, A, P);
    return mj * fma(q * q, A, P);
}

template <int NK>
__device__ __forceinline__ void psi_visit(PsiLds &lds, double xr, double yr, double zr, float px,
                                          float py, float pz, double Hi, double invHi, float cand2,
                                          double &ps)
{
    const int lane = threadIdx.x & 63;
    uint64_t mine = 0;   // bit jj: the pair with jj may be within H_i
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        unsigned list = 0;
#pragma unroll 8
        for (int jj = 31; jj >= 0; --jj) {
            const float4 p = lds.f[32 * h + jj];
            const float dx = p.x - px, dy = p.y - py, dz = p.z - pz;
            const bool in = fmaf(dx, dx, fmaf(dy, dy, dz * dz)) <= cand2;
            list = list + list + (in ? 1u : 0u);
        }
        mine |= (uint64_t)list << (32 * h);
    }
    const unsigned count = (unsigned)__builtin_popcountll(mine);
    unsigned at, total;
    list_places(count, at, total);
    if (total > (unsigned)NSOFT) {
        while (mine) {
            const int jj = __builtin_ctzll(mine);
            mine &= mine - 1;
            const double4 p = lds.p[jj];
            ps += psi_pair<NK>(p.x - xr, p.y - yr, p.z - zr, Hi, invHi, p.w);
        }
        return;
    }
    for (unsigned k = at; mine; ++k) {
        const int jj = __builtin_ctzll(mine);
        mine &= mine - 1;
        lds.list[k] = (uint16_t)(lane << 6 | jj);
    }
    for (unsigned b0 = 0; b0 < total; b0 += 64) {
        wave_lds_sync();
        const unsigned e = min(b0 + (unsigned)lane, total - 1);
        const int il = lds.list[e] >> 6, jj = lds.list[e] & 63;
        const double4 p = lds.p[jj];
        lds.res[lane] = psi_pair<NK>(p.x - __shfl(xr, il, 64), p.y - __shfl(yr, il, 64),
                                     p.z - __shfl(zr, il, 64), __shfl(Hi, il, 64),
                                     __shfl(invHi, il, 64), p.w);
        wave_lds_sync();
        const unsigned hi = min(at + count, b0 + 64);
        for (unsigned k = max(at, b0); k < hi; ++k) ps += lds.res[k - b0];
    }
}

template <int NK>
__global__ __launch_bounds__(64) void k_psi_only(PairArgs a)
{
    __shared__ PsiLds lds;
    const int lane = threadIdx.x;
    const unsigned ng = (unsigned)a.ngroups;
    const int64_t gbase = (int64_t)(blockIdx.x % ng) * 64;
    const int part = (int)(blockIdx.x / ng);
    const int64_t io = min(gbase + 32, a.ni - 1);
    const double Ox = a.i.x[io], Oy = a.i.y[io], Oz = a.i.z[io];
    const bool valid = gbase + lane < a.ni;
    const int64_t i = valid ? gbase + lane : a.ni - 1;
    const double xr = a.i.x[i] - Ox, yr = a.i.y[i] - Oy, zr = a.i.z[i] - Oz;
    const double Hi = fabs(a.i.Hs[i]), invHi = 1.0 / Hi, hi2 = Hi * Hi;
    float bl[3] = {(float)xr, (float)yr, (float)zr}, bh[3] = {bl[0], bl[1], bl[2]};
    for (int c = 0; c < 3; ++c) {
        bl[c] = wave_min(bl[c]);
        bh[c] = wave_max(bh[c]);
    }
    // only side i matters for psi: a chunk farther from the group's box than the
    // wave's largest H_i, or from a lane's particle than its own, holds no pair of
    // theirs.  That of a pair is off in FP32 like that to a box (box_slack).
    const float px = (float)xr, py = (float)yr, pz = (float)zr;
    const float slack = box_slack(px, py, pz);
    const float cand = (float)Hi * (1.0f + 2.0e-6f) + slack;
    const float cand2 = cand * cand;
    const float lim = wave_max((float)Hi) * (1.0f + 2.0e-6f) + wave_max(slack);
    const float lim2 = lim * lim;
    double ps = 0.0;
    // part p has every jsplit-th chunk (jsplit a power of two), of the tiles
    // that hold one of them
    const int other = a.jsplit - 1;
    for (int tb = 0; tb < a.ntiles; tb += 64) {
        const int tl = min(tb + lane, a.ntiles - 1);
        uint64_t tiles = __ballot(tb + lane < a.ntiles &&
                                  ((tl * CHUNKS ^ part) & other & ~(CHUNKS - 1)) == 0 &&
                                  box_dist2(a.tiles[tl], Ox, Oy, Oz, bl, bh) <= lim2);
        for (; tiles; tiles &= tiles - 1) {
            const int64_t c0 = (int64_t)(tb + __builtin_ctzll(tiles)) * CHUNKS;
            unsigned bits = (unsigned)__ballot(
                lane < CHUNKS && ((lane ^ part) & other & (CHUNKS - 1)) == 0 &&
                box_dist2(a.chunks[c0 + (lane & (CHUNKS - 1))], Ox, Oy, Oz, bl, bh) <= lim2);
            for (; bits; bits &= bits - 1) {
                // the group's box and largest H pass many chunks that no lane's
                // own particle reaches
                const TileMeta &cm = a.chunks[c0 + __builtin_ctz(bits)];
                const float gx = fmaxf(0.0f, fmaxf((float)(cm.lo[0] - Ox) - px, px - (float)(cm.hi[0] - Ox)));
                const float gy = fmaxf(0.0f, fmaxf((float)(cm.lo[1] - Oy) - py, py - (float)(cm.hi[1] - Oy)));
                const float gz = fmaxf(0.0f, fmaxf((float)(cm.lo[2] - Oz) - pz, pz - (float)(cm.hi[2] - Oz)));
                if (!__ballot(fmaf(gx, gx, fmaf(gy, gy, gz * gz)) <= cand2)) continue;
                const int64_t j = (c0 + __builtin_ctz(bits)) * TC + lane;
                wave_lds_sync();
                const double jx = a.j.x[j] - Ox, jy = a.j.y[j] - Oy, jz = a.j.z[j] - Oz;
                lds.p[lane] = make_double4(jx, jy, jz, a.j.m[j]);
                lds.f[lane] = make_float4((float)jx, (float)jy, (float)jz, 0.0f);
                wave_lds_sync();
                psi_visit<NK>(lds, xr, yr, zr, px, py, pz, Hi, invHi, cand2, ps);
            }
        }
    }
    if (valid) a.psipart[(int64_t)part * a.ni + i] = ps;
}

// Fixed-order sum of the parts, scattered to input order (0 for point
// particles).
__global__ __launch_bounds__(256) void k_psi_reduce(PairArgs a)
{
    const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
    if (i >= a.ni) return;
    double ps = 0.0;
    for (int p = 0; p < a.jsplit; ++p) ps += a.psipart[(int64_t)p * a.ni + i];
    const double Hs = a.i.Hs[i];
    a.psi[(int64_t)a.i.idx[i] - a.ibeg] = Hs > 0.0 ? -2.0 / (Hs * Hs) * ps : 0.0;
}

// Fixed-order FP64 sum of the j-partition partials, scattered to input order:
// a block takes 64 particles of one sum (blockIdx.y: ax, ay, az, pot, psi),
// each of its waves a quarter of the partitions, eight loads in flight.
__global__ __launch_bounds__(256) void k_reduce_partials(PairArgs a)
{
    __shared__ double s_sum[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t i = blockIdx.x * (int64_t)64 + lane;
    const int c = blockIdx.y;
    const int64_t step = c < 4 ? 4 * a.ni : a.ni;
    double s = 0.0;
    if (i < a.ni) {
        const double *p = c < 4 ? a.partial + c * a.ni + i : a.psipart + i;
        const int end = a.jsplit * (w + 1) / 4;
#pragma unroll 8
        for (int jp = a.jsplit * w / 4; jp < end; ++jp) s += p[jp * step];
    }
    s_sum[w][lane] = s;
    __syncthreads();
    if (w != 0 || i >= a.ni) return;
    double *out = c == 0 ? a.ax : (c == 1 ? a.ay : (c == 2 ? a.az : (c == 3 ? a.pot : a.psi)));
    out[(int64_t)a.i.idx[i] - a.ibeg] = s + s_sum[1][lane] + s_sum[2][lane] + s_sum[3][lane];
}

// ============================================================= batch kernels
template <int WG, int IPL>
__device__ __forceinline__ Block batch_block(const BatchArgs &a, int item)
{
    const int2 it = a.items[item];
    const BatchSet st = a.sets[it.x];
    const int ib = it.y / st.jsplit, jp = it.y - ib * st.jsplit;
    const int64_t pad = (int64_t)st.ntiles * TJ;
    Block b;
    b.ibase = st.pofs + (int64_t)ib * WG * IPL;
    b.iend = st.pofs + st.n;
    b.t0 = st.tile0 + jp;
    b.t1 = st.tile0 + st.ntiles;
    b.tstep = st.jsplit;
    b.fbase = st.tile0;
    b.fstride = st.ntiles;
    b.flags = a.nearflag + st.flagofs + (int64_t)ib * (WG / 64) * st.ntiles;
    // partition jp's slab; slot i of the set sits at [i - pofs] (partofs >=
    // pofs, so the base stays inside the buffer)
    b.part = a.partial + (st.partofs - st.pofs) + (int64_t)jp * 4 * pad;
    b.pstride = pad;
    return b;
}

// Persistent far kernel over a batch: every workgroup takes the next
// (set, i-block, j-partition) item from the queue until the queue is empty,
// so every workgroup reaches the exit once all items are taken.
template <int WG, int IPL, bool FP64, int NK>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(IPL == 1 && !FP64 ? 7 : 1)))
void k_far_batch(BatchArgs a)
{
    // one TS-entry FP64 tile, or the FP32 hi stage followed by the FP64 stage
    __shared__ double4 s_buf[TS + TS / 2];
    float4 *s_hi = reinterpret_cast<float4 *>(s_buf);
    double4 *s_p = s_buf + TS / 2;
    __shared__ NearSlice s_near[FP64 ? 1 : WG / 64];
    __shared__ int s_item;
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) s_item = (int)atomicAdd(a.counter, 1u);
        __syncthreads();
        const int item = s_item;
        if (item >= a.nitems) break;
        const Block b = batch_block<WG, IPL>(a, item);
        if (FP64)
            far_block_fp64<WG, IPL>(a.j, a.j, a.tiles, a.chunks, b, a.stats, s_buf);
        else
            far_block_fp32c<WG, IPL, NK, true>(a.j, a.j, a.tiles, a.chunks, b, a.stats, s_hi,
                                               s_p, s_near);
    }
}

template <int IPL, bool FAST, int NK>
__global__ __launch_bounds__(64 * NEAR_WAVES) void k_near_batch(BatchArgs a)
{
    __shared__ NearLds lds;
    __shared__ double s_red[(NEAR_WAVES - 1) * 4 * IPL * 64];
    const int64_t gg = blockIdx.x;
    // the set this group belongs to (sets are ordered by group offset)
    int lo = 0, hi = a.nsets - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (a.sets[mid].gofs <= gg) lo = mid;
        else hi = mid - 1;
    }
    const BatchSet st = a.sets[lo];
    const int64_t lg = gg - st.gofs;
    Group g;
    g.gbase = st.pofs + lg * (64 * IPL);
    g.iend = st.pofs + st.n;
    g.t0 = st.tile0;
    g.t1 = st.tile0 + st.ntiles;
    g.flags = a.nearflag + st.flagofs + lg * st.ntiles;
    // added to the set's first partition slab (after the far kernel)
    g.part = a.partial + (st.partofs - st.pofs);
    g.pstride = (int64_t)st.ntiles * TJ;
    if (g.gbase >= g.iend || !group_has_near(g)) return;
    near_group<IPL, FAST, NK>(a.j, a.j, g, lds, s_red);
}

// Sum the partition slabs of each slot in a fixed order (partition 0
// first) and scatter the sums back to input order.
__global__ __launch_bounds__(256) void k_reduce_batch(BatchArgs a)
{
    const int64_t s = blockIdx.x * (int64_t)256 + threadIdx.x;
    if (s >= a.padded) return;
    const int o = a.j.idx[s];
    if (o < 0) return;   // padding
    // the set of slot s (sets are ordered by first slot)
    int lo = 0, hi = a.nsets - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (a.sets[mid].pofs <= s) lo = mid;
        else hi = mid - 1;
    }
    const BatchSet st = a.sets[lo];
    const int64_t pad = (int64_t)st.ntiles * TJ;
    const double *p = a.partial + st.partofs + (s - st.pofs);
    double v[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) v[c] = p[c * pad];
    for (int q = 1; q < st.jsplit; ++q) {
        p += 4 * pad;
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] += p[c * pad];
    }
    a.ax[o] = v[0];
    a.ay[o] = v[1];
    a.az[o] = v[2];
    a.pot[o] = v[3];
}

inline dim3 grid_of(const PairArgs &a) { return dim3((unsigned)a.niblocks * (unsigned)a.jsplit); }

}  // namespace

#define SG_FAR(KERNEL, WG, IPL)                                                        \
    if (wg == WG && a.ipl == IPL) {                                                    \
        hipLaunchKernelGGL((KERNEL<WG, IPL>), grid_of(a), dim3(WG), 0, s, a);          \
        return hipGetLastError();                                                      \
    }

template <int WG, int IPL>
static hipError_t far_fused_launch(const PairArgs &a, hipStream_t s)
{
    switch (a.nkernel) {
    case 0: hipLaunchKernelGGL((k_far_fp32c<WG, IPL, 0>), grid_of(a), dim3(WG), 0, s, a); break;
    case 1: hipLaunchKernelGGL((k_far_fp32c<WG, IPL, 1>), grid_of(a), dim3(WG), 0, s, a); break;
    case 2: hipLaunchKernelGGL((k_far_fp32c<WG, IPL, 2>), grid_of(a), dim3(WG), 0, s, a); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <bool PSI>
static hipError_t wave_launch(const PairArgs &a, hipStream_t s)
{
    const dim3 grid((unsigned)((a.ni + TC - 1) / TC) * (unsigned)a.jsplit), block(64);
    switch (a.nkernel) {
    case 0: hipLaunchKernelGGL((k_pair_wave<0, PSI>), grid, block, 0, s, a); break;
    case 1: hipLaunchKernelGGL((k_pair_wave<1, PSI>), grid, block, 0, s, a); break;
    case 2: hipLaunchKernelGGL((k_pair_wave<2, PSI>), grid, block, 0, s, a); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// FP32C: one wave per 64 i and j partition (a.wave), else the fused far kernel
// (no near kernel follows either), or, with the grad-h term, the split far
// kernel with one i per lane.  FP64: the far kernel.
hipError_t launch_pair_far(int precision, const PairArgs &a, int wg, hipStream_t s)
{
    if (a.ni <= 0) return hipSuccess;
    if (precision == 0 && a.wave) return a.psi ? wave_launch<true>(a, s) : wave_launch<false>(a, s);
    if (precision == 0 && a.psi) {
        if (a.ipl != 1) return hipErrorInvalidConfiguration;
        switch (wg) {
        case 64: hipLaunchKernelGGL((k_far_fp32c_split<64>), grid_of(a), dim3(64), 0, s, a); break;
        case 128: hipLaunchKernelGGL((k_far_fp32c_split<128>), grid_of(a), dim3(128), 0, s, a); break;
        case 256: hipLaunchKernelGGL((k_far_fp32c_split<256>), grid_of(a), dim3(256), 0, s, a); break;
        default: return hipErrorInvalidConfiguration;
        }
        return hipGetLastError();
    }
    if (precision == 0) {
        if (wg == 64 && a.ipl == 1) return far_fused_launch<64, 1>(a, s);
        if (wg == 64 && a.ipl == 2) return far_fused_launch<64, 2>(a, s);
        if (wg == 128 && a.ipl == 1) return far_fused_launch<128, 1>(a, s);
        if (wg == 128 && a.ipl == 2) return far_fused_launch<128, 2>(a, s);
        if (wg == 256 && a.ipl == 1) return far_fused_launch<256, 1>(a, s);
        if (wg == 256 && a.ipl == 2) return far_fused_launch<256, 2>(a, s);
    } else {
        SG_FAR(k_far_fp64, 64, 1) SG_FAR(k_far_fp64, 64, 2)
        SG_FAR(k_far_fp64, 128, 1) SG_FAR(k_far_fp64, 128, 2)
        SG_FAR(k_far_fp64, 256, 1) SG_FAR(k_far_fp64, 256, 2)
    }
    return hipErrorInvalidConfiguration;
}

template <int IPL>
static void near_launch(const PairArgs &a, dim3 grid, dim3 block, hipStream_t s)
{
    switch (a.nkernel) {
    case 0: hipLaunchKernelGGL((k_near<IPL, false, 0>), grid, block, 0, s, a); break;
    case 1: hipLaunchKernelGGL((k_near<IPL, false, 1>), grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL((k_near<IPL, false, 2>), grid, block, 0, s, a); break;
    }
}

template <bool FAST>
static void near_psi_launch(const PairArgs &a, dim3 grid, dim3 block, hipStream_t s)
{
    switch (a.nkernel) {
    case 0: hipLaunchKernelGGL((k_near_psi<FAST, 0>), grid, block, 0, s, a); break;
    case 1: hipLaunchKernelGGL((k_near_psi<FAST, 1>), grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL((k_near_psi<FAST, 2>), grid, block, 0, s, a); break;
    }
}

// The near kernel of the FP64 pass and of the grad-h pass; the FP32C
// forward pass has none (its far kernel takes the near chunks).
hipError_t launch_pair_near(int precision, const PairArgs &a, hipStream_t s)
{
    if (a.ni <= 0) return hipSuccess;
    if (a.nkernel < 0 || a.nkernel > 2) return hipErrorInvalidValue;
    if (precision == 0 && a.wave) return hipSuccess;   // its waves take the near chunks
    const dim3 grid((unsigned)(a.ngroups * a.jsplit)), block(64 * NEAR_WAVES);
    if (a.psi) {
        if (a.ipl != 1) return hipErrorInvalidConfiguration;
        hipError_t e = launch_fill_zero_int(reinterpret_cast<int *>(a.psipart),
                                            (int)(2 * (int64_t)a.jsplit * a.ni), s);
        if (e != hipSuccess) return e;
        if (precision == 0) near_psi_launch<true>(a, grid, block, s);
        else near_psi_launch<false>(a, grid, block, s);
        return hipGetLastError();
    }
    if (precision == 0) return hipSuccess;
    switch (a.ipl) {
    case 1: near_launch<1>(a, grid, block, s); break;
    case 2: near_launch<2>(a, grid, block, s); break;
    default: return hipErrorInvalidConfiguration;
    }
    return hipGetLastError();
}

bool pair_config_supported(int precision, int wg, int ipl)
{
    (void)precision;
    return (wg == 64 || wg == 128 || wg == 256) && (ipl == 1 || ipl == 2);
}

hipError_t launch_psi_only(const PairArgs &a, hipStream_t s)
{
    if (a.ni <= 0) return hipSuccess;
    const dim3 grid((unsigned)a.ngroups * (unsigned)a.jsplit), block(64);
    switch (a.nkernel) {
    case 0: hipLaunchKernelGGL((k_psi_only<0>), grid, block, 0, s, a); break;
    case 1: hipLaunchKernelGGL((k_psi_only<1>), grid, block, 0, s, a); break;
    case 2: hipLaunchKernelGGL((k_psi_only<2>), grid, block, 0, s, a); break;
    default: return hipErrorInvalidValue;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_psi_reduce, dim3((unsigned)((a.ni + 255) / 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_sym_rest(const SymArgs &a, hipStream_t s)
{
    // as many waves as there can be segments; those past the last one end at once
    const dim3 grid((unsigned)(SYM_SEGS + a.nchunks)), block(64);
#define SG_REST(k, nk, fp64, psi) \
    case k: hipLaunchKernelGGL((k_sym_rest<nk, fp64, psi>), grid, block, 0, s, a); break;
    switch (a.nkernel + (a.fp64 ? 3 : 0) + (a.psi ? 6 : 0)) {
        SG_REST(0, 0, false, false) SG_REST(1, 1, false, false) SG_REST(2, 2, false, false)
        SG_REST(3, 0, true, false) SG_REST(4, 1, true, false) SG_REST(5, 2, true, false)
        SG_REST(6, 0, false, true) SG_REST(7, 1, false, true) SG_REST(8, 2, false, true)
        SG_REST(9, 0, true, true) SG_REST(10, 1, true, true) SG_REST(11, 2, true, true)
    default: return hipErrorInvalidValue;
    }
#undef SG_REST
    return hipGetLastError();
}

hipError_t launch_reduce_partials(const PairArgs &a, hipStream_t s)
{
    if (a.ni <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_reduce_partials, dim3((unsigned)((a.ni + 63) / 64), a.psi ? 5 : 4),
                       dim3(256), 0, s, a);
    return hipGetLastError();
}

// ------------------------------------------------------------ batch launches
// FP32C batches run the fused far kernel (one instantiation per softening
// kernel NK); FP64 batches the plain far kernel (NK = 0) and then the near
// kernel.
template <int WG, int IPL, bool FP64, int NK>
static hipError_t far_batch_launch(const BatchArgs &a, int nwg, hipStream_t s)
{
    hipLaunchKernelGGL((k_far_batch<WG, IPL, FP64, NK>), dim3(nwg), dim3(WG), 0, s, a);
    return hipGetLastError();
}

template <int WG, int IPL, bool FP64, int NK>
static int far_batch_resident(int device)
{
    int per_cu = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_far_batch<WG, IPL, FP64, NK>, WG,
                                                     0) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
        return 0;
    return per_cu * cus;
}

template <int WG, int IPL>
static int far_batch_one(int precision, int nk, const BatchArgs &a, int nwg, hipStream_t s,
                         bool resident_only, int device)
{
    if (precision != 0)
        return resident_only ? far_batch_resident<WG, IPL, true, 0>(device)
                             : (int)far_batch_launch<WG, IPL, true, 0>(a, nwg, s);
    switch (nk) {
    case 0:
        return resident_only ? far_batch_resident<WG, IPL, false, 0>(device)
                             : (int)far_batch_launch<WG, IPL, false, 0>(a, nwg, s);
    case 1:
        return resident_only ? far_batch_resident<WG, IPL, false, 1>(device)
                             : (int)far_batch_launch<WG, IPL, false, 1>(a, nwg, s);
    default:
        return resident_only ? far_batch_resident<WG, IPL, false, 2>(device)
                             : (int)far_batch_launch<WG, IPL, false, 2>(a, nwg, s);
    }
}

static int far_batch_dispatch(int precision, int nk, const BatchArgs &a, int wg, int ipl, int nwg,
                              hipStream_t s, bool resident_only, int device)
{
    if (wg == 64 && ipl == 1) return far_batch_one<64, 1>(precision, nk, a, nwg, s, resident_only, device);
    if (wg == 64 && ipl == 2) return far_batch_one<64, 2>(precision, nk, a, nwg, s, resident_only, device);
    if (wg == 128 && ipl == 1) return far_batch_one<128, 1>(precision, nk, a, nwg, s, resident_only, device);
    if (wg == 128 && ipl == 2) return far_batch_one<128, 2>(precision, nk, a, nwg, s, resident_only, device);
    if (wg == 256 && ipl == 1) return far_batch_one<256, 1>(precision, nk, a, nwg, s, resident_only, device);
    if (wg == 256 && ipl == 2) return far_batch_one<256, 2>(precision, nk, a, nwg, s, resident_only, device);
    return resident_only ? 0 : (int)hipErrorInvalidConfiguration;
}

int batch_resident_workgroups(int precision, int nkernel, int wg, int ipl, int device)
{
    BatchArgs dummy{};
    return far_batch_dispatch(precision, nkernel, dummy, wg, ipl, 0, nullptr, true, device);
}

bool batch_config_supported(int wg, int ipl)
{
    return (wg == 64 || wg == 128 || wg == 256) && (ipl == 1 || ipl == 2);
}

template <int IPL>
static void near_batch_launch(const BatchArgs &a, dim3 grid, dim3 block, hipStream_t s)
{
    switch (a.nkernel) {
    case 0: hipLaunchKernelGGL((k_near_batch<IPL, false, 0>), grid, block, 0, s, a); break;
    case 1: hipLaunchKernelGGL((k_near_batch<IPL, false, 1>), grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL((k_near_batch<IPL, false, 2>), grid, block, 0, s, a); break;
    }
}

hipError_t launch_batch(int precision, const BatchArgs &a, int wg, int ipl, int nwg, hipStream_t s)
{
    if (a.nkernel < 0 || a.nkernel > 2) return hipErrorInvalidValue;
    if (a.padded <= 0) return hipSuccess;
    hipError_t e = launch_fill_zero_int((int *)a.counter, 1, s);
    if (e != hipSuccess) return e;
    e = (hipError_t)far_batch_dispatch(precision, a.nkernel, a, wg, ipl, nwg, s, false, 0);
    if (e != hipSuccess) return e;
    const dim3 block(64 * NEAR_WAVES), grid((unsigned)a.ngroups);
    if (precision != 0 && a.ngroups > 0) {
        if (ipl == 1) near_batch_launch<1>(a, grid, block, s);
        else near_batch_launch<2>(a, grid, block, s);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k_reduce_batch, dim3((unsigned)((a.padded + 255) / 256)), dim3(256), 0, s,
                       a);
    return hipGetLastError();
}

}  // namespace sg
