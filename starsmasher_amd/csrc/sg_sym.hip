// sg_sym.hip -- far pairs of a whole set, each unordered pair evaluated once
// (gfx950).
//
// A pair of far, Newtonian particles contributes m_j r^-3 (x_j - x_i) to i
// and -m_i r^-3 (x_j - x_i) to j: one difference, one r^2 and one
// v_rsq_f32 serve both.  Per unordered pair that is 18 FP32 VALU operations
// and one v_rsq_f32 against 26 and 2 for the two ordered pairs.
//
//   * k_sym_classify marks the pairs of 64-particle chunks that qualify: all
//     pairs Newtonian by the box test, far enough from the row chunk, relative
//     to its own half-diagonal, for FP32 differences of positions rounded
//     relative to its centre, and not closer than SCALED_MIN of the set's
//     extent, which bounds the powers of 1/r below.  Every other (chunk, chunk) visit is
//     left to the ordered rest kernel (sg_direct.hip).
//   * k_sym evaluates the marked pairs.  A wave holds a 64-particle row chunk
//     (the i side) and meets 64-particle column chunks (the j side); its lanes
//     form a 4 x 16 grid, lane (p, q) holding i = 16 p .. 16 p + 15 and
//     j = q, q + 16, q + 32, q + 48 in registers with their sums, so the pair
//     loop reads no memory and moves nothing between lanes.  The j sums of a
//     chunk pair are reduced over p (two register-half swaps), the i sums of
//     four chunk pairs over q.
//   * Positions and masses are scaled by powers of two (the set's extent and
//     largest mass become order one; the reduce kernel undoes it), so that r^-3
//     stays in the FP32 range in any units: at most 2^60 (SCALED_MIN), and the
//     gradient's terms in r^-4 2^84 times the cotangents.
//   * Sums go to FP64 after at most 16 sequential FP32 additions and a tree
//     over the lanes.
//   * Work items are pairs of superblocks.  Every (superblock, superblock)
//     pair has partial-sum slabs of its own, added in a fixed order by the
//     reduce kernel: results do not depend on scheduling, no atomics between
//     workgroups.
#include "sg_internal.h"
#include "sg_device.h"
#include "sg_lanes.h"

namespace sg {
namespace {

constexpr int NP = 4, NQ = 16;         // lane grid: i groups x j groups
constexpr int IA = TC / NP;            // i per lane
constexpr int JB = TC / NQ;            // j per lane
constexpr int JC = 4;                  // column chunks a wave owns at a time
constexpr double SCALED_MIN = 0x1p-20; // about a cell of the curve: rarely the nearer bound
static_assert(NP * NQ == 64 && IA == 16 && JB == 4, "lane grid");

// ------------------------------------------------------------ chunk pairs
// FP32 chunk boxes relative to the centre of the set's box, rounded outwards
// (a gap computed from them never exceeds the true one): {lo, H}, {hi, the
// squared half-diagonal}.
__global__ __launch_bounds__(256) void k_sym_boxes(SymArgs a)
{
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= a.nchunks) return;
    const TileMeta m = a.chunks[c];
    if (a.sets) a.bbox += 8 * (int64_t)a.setof[c];
    float lo[3], hi[3], rho2 = 0.0f;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const double o = 0.5 * (a.bbox[k] + a.bbox[3 + k]);
        lo[k] = __double2float_rd(m.lo[k] - o);
        hi[k] = __double2float_ru(m.hi[k] - o);
        const float h = 0.5f * (float)(m.hi[k] - m.lo[k]);
        rho2 = fmaf(h, h, rho2);
    }
    a.boxes[2 * c] = make_float4(lo[0], lo[1], lo[2], (float)m.maxH);
    a.boxes[2 * c + 1] = make_float4(hi[0], hi[1], hi[2], rho2);
}

// One wave per CROWS row chunks: the bits of the rows, 64 column chunks at a
// time, and the number of unset ones.  The half-diagonal is that of the lower
// chunk index, the row in k_sym, for both (ci, cj) and (cj, ci), so the bit
// matrix is symmetric.
constexpr int CROWS = 4;
static_assert(CHUNKS % CROWS == 0, "a tile's chunks are whole groups of rows");
__global__ __launch_bounds__(256) void k_sym_classify(SymArgs a)
{
    const int lane = threadIdx.x & 63;
    int r0 = uniform_i((int)(blockIdx.x * 4 + (threadIdx.x >> 6)) * CROWS);
    if (r0 >= a.nchunks) return;
    if (a.sets) {   // sets begin at a tile, so CROWS rows share one
        const int set = a.setof[r0];
        r0 -= uniform_i(a.sets[set].chunk0);
        a = sym_view(a, set);
    }
    float4 rl[CROWS], rh[CROWS];
    int rest[CROWS];
#pragma unroll
    for (int r = 0; r < CROWS; ++r) {
        const int ci = min(r0 + r, a.nchunks - 1);
        rl[r] = a.boxes[2 * ci];
        rh[r] = a.boxes[2 * ci + 1];
        rest[r] = a.nchunks;
    }
    const float wide = a.fp64 ? 0.0f : WIDE_K * WIDE_K;
    // least squared distance (FP32 overflow: the largest, which an infinite d2 passes)
    const double least = a.fp64 ? 0.0 : SCALED_MIN / a.bbox[6];
    const float least2 = (float)fmin(least * least, 3.0e38);
    for (int w = 0; w < a.words; ++w) {
        const int cj = w * 64 + lane;
        const int cc = min(cj, a.nchunks - 1);
        const float4 cl = a.boxes[2 * cc], ch = a.boxes[2 * cc + 1];
#pragma unroll
        for (int r = 0; r < CROWS; ++r) {
            const int ci = r0 + r;
            const float gx = fmaxf(0.0f, fmaxf(cl.x - rh[r].x, rl[r].x - ch.x));
            const float gy = fmaxf(0.0f, fmaxf(cl.y - rh[r].y, rl[r].y - ch.y));
            const float gz = fmaxf(0.0f, fmaxf(cl.z - rh[r].z, rl[r].z - ch.z));
            const float d2 = fmaf(gx, gx, fmaf(gy, gy, gz * gz));
            const float hm = fmaxf(cl.w, rl[r].w);
            const float rho2 = cj < ci ? ch.w : rh[r].w;
            const bool ok = cj < a.nchunks && cj != ci &&
                            d2 > fmaxf(fmaxf(hm * hm, wide * rho2), least2) * (1.0f + FAR_MARGIN);
            const uint64_t bits = __ballot(ok);
            rest[r] -= __builtin_popcountll(bits);
            if (ci < a.nchunks && lane == 0) a.sym[(int64_t)ci * a.words + w] = bits;
        }
    }
#pragma unroll
    for (int r = 0; r < CROWS; ++r) {
        if (lane != 0) continue;
        if (r0 + r < a.nchunks) a.seg[r0 + r] = rest[r];
        else if (a.sets) a.seg[r0 + r] = 0;   // the rest of the set's last tile: padding only
    }
}

// Cuts each row's unset bits into segments of at most `len` visits, len chosen
// so that at most SYM_SEGS + nchunks segments result: a.seg[c] becomes the
// first segment of row c, a.seg[nchunks] their number, a.seg[nchunks + 1] len.
// One workgroup.
__global__ __launch_bounds__(1024) void k_sym_segments(SymArgs a)
{
    __shared__ int64_t s_sum[1024];
    const int t = threadIdx.x;
    const int per = (a.nchunks + 1023) / 1024;
    const int c0 = min(t * per, a.nchunks), c1 = min(c0 + per, a.nchunks);
    int64_t v = 0;
    for (int c = c0; c < c1; ++c) v += a.seg[c];
    s_sum[t] = v;
    __syncthreads();
    for (int o = 512; o > 0; o >>= 1) {
        if (t < o) s_sum[t] += s_sum[t + o];
        __syncthreads();
    }
    const int len = (int)max((int64_t)SYM_SEG_MIN, (s_sum[0] + SYM_SEGS - 1) / SYM_SEGS);
    __syncthreads();
    int n = 0;
    for (int c = c0; c < c1; ++c) n += (a.seg[c] + len - 1) / len;
    s_sum[t] = n;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
        const int64_t u = t >= o ? s_sum[t - o] : 0;
        __syncthreads();
        s_sum[t] += u;
        __syncthreads();
    }
    int at = (int)s_sum[t] - n;
    for (int c = c0; c < c1; ++c) {
        const int k = (a.seg[c] + len - 1) / len;
        a.seg[c] = at;
        at += k;
    }
    if (t == 1023) {
        a.seg[a.nchunks] = at;
        a.segtot[0] = at;
        a.segtot[1] = len;
    }
}

// ------------------------------------------------------------- pair groups
// Four unordered pairs (one i, four j) as one block of instructions.  What
// the block fixes, and a compiler left alone does not:
//   * the four v_rsq_f32 are issued back to back at raised wave priority.
//     A v_rsq_f32 takes 8 cycles and issues alone, while two waves of a SIMD
//     issue other FP32 instructions together (2.2 cycles each) as long as they
//     stay in step; at equal priority the wave that is first past its v_rsq_f32
//     runs ahead by itself and joint issue is lost (measured on this body: 79
//     cycles a pair without stalls, 58-65 with the compiler's waits, 48.8 with
//     the priority, against 48 by instruction count);
//   * the three register sources of an FMA never have the same parity (odd
//     or even number), which would also forbid joint issue (4.1 cycles, not
//     2.2): differences and r^-1 sit in even registers, the force factors in
//     odd ones, and masses are the fourth (odd) register of a loaded quad.
#define SYM_DIFF(k, dx, dy, dz, r)                                             \
    "v_sub_f32_e32 v" dx ", %[xj" k "], %[xi]\n\t"                             \
    "v_sub_f32_e32 v" dy ", %[yj" k "], %[yi]\n\t"                             \
    "v_sub_f32_e32 v" dz ", %[zj" k "], %[zi]\n\t"                             \
    "v_mul_f32_e32 v" r ", v" dz ", v" dz "\n\t"                               \
    "v_fmac_f32_e32 v" r ", v" dy ", v" dy "\n\t"                              \
    "v_fmac_f32_e32 v" r ", v" dx ", v" dx "\n\t"
#define SYM_RSQ(ri, r) "v_rsq_f32_e32 v" ri ", v" r "\n\t"
#define SYM_SUM_I(k, dx, dy, dz, ri, f, h)                                     \
    "v_mul_f32_e32 v" f ", v" ri ", v" ri "\n\t"                               \
    "v_mul_f32_e32 v" f ", v" f ", v" ri "\n\t"                                \
    "v_mul_f32_e32 v" h ", %[mj" k "], v" f "\n\t"                             \
    "v_mul_f32_e32 v" f ", %[mi], v" f "\n\t"                                  \
    "v_fmac_f32_e32 %[ax], v" h ", v" dx "\n\t"                                \
    "v_fmac_f32_e32 %[ay], v" h ", v" dy "\n\t"                                \
    "v_fmac_f32_e32 %[az], v" h ", v" dz "\n\t"                                \
    "v_fmac_f32_e32 %[ap], %[mj" k "], v" ri "\n\t"
#define SYM_SUM_J(op, k, dx, dy, dz, ri, f)                                    \
    op " %[bx" k "], v" f ", v" dx "\n\t"                                      \
    op " %[by" k "], v" f ", v" dy "\n\t"                                      \
    op " %[bz" k "], v" f ", v" dz "\n\t"                                      \
    op " %[bp" k "], %[mi], v" ri "\n\t"
// even: dx, dy, dz, r^-1; odd: r^2 then f, h (the j side's force factor)
#define SYM_GROUP(op)                                                          \
    SYM_DIFF("0", "8", "10", "12", "9") SYM_DIFF("1", "16", "18", "20", "17")  \
    SYM_DIFF("2", "24", "26", "28", "25") SYM_DIFF("3", "32", "34", "36", "33") \
    "s_setprio 3\n\t"                                                          \
    SYM_RSQ("14", "9") SYM_RSQ("22", "17") SYM_RSQ("30", "25") SYM_RSQ("38", "33") \
    "s_setprio 0\n\t"                                                          \
    SYM_SUM_I("0", "8", "10", "12", "14", "9", "11")                           \
    SYM_SUM_J(op, "0", "8", "10", "12", "14", "9")                             \
    SYM_SUM_I("1", "16", "18", "20", "22", "17", "19")                         \
    SYM_SUM_J(op, "1", "16", "18", "20", "22", "17")                           \
    SYM_SUM_I("2", "24", "26", "28", "30", "25", "27")                         \
    SYM_SUM_J(op, "2", "24", "26", "28", "30", "25")                           \
    SYM_SUM_I("3", "32", "34", "36", "38", "33", "35")                         \
    SYM_SUM_J(op, "3", "32", "34", "36", "38", "33")
#define SYM_J_SUMS(c)                                                          \
    [bx0] c(j.s[0][0]), [by0] c(j.s[0][1]), [bz0] c(j.s[0][2]), [bp0] c(j.s[0][3]), \
    [bx1] c(j.s[1][0]), [by1] c(j.s[1][1]), [bz1] c(j.s[1][2]), [bp1] c(j.s[1][3]), \
    [bx2] c(j.s[2][0]), [by2] c(j.s[2][1]), [bz2] c(j.s[2][2]), [bp2] c(j.s[2][3]), \
    [bx3] c(j.s[3][0]), [by3] c(j.s[3][1]), [bz3] c(j.s[3][2]), [bp3] c(j.s[3][3])
#define SYM_INPUTS                                                             \
    [xi] "v"(xi.x), [yi] "v"(xi.y), [zi] "v"(xi.z), [mi] "v"(xi.w),            \
    [xj0] "v"(j.x[0].x), [yj0] "v"(j.x[0].y), [zj0] "v"(j.x[0].z), [mj0] "v"(j.x[0].w), \
    [xj1] "v"(j.x[1].x), [yj1] "v"(j.x[1].y), [zj1] "v"(j.x[1].z), [mj1] "v"(j.x[1].w), \
    [xj2] "v"(j.x[2].x), [yj2] "v"(j.x[2].y), [zj2] "v"(j.x[2].z), [mj2] "v"(j.x[2].w), \
    [xj3] "v"(j.x[3].x), [yj3] "v"(j.x[3].y), [zj3] "v"(j.x[3].z), [mj3] "v"(j.x[3].w)
#define SYM_TEMPS                                                              \
    "v8", "v9", "v10", "v11", "v12", "v14", "v16", "v17", "v18", "v19", "v20", \
    "v22", "v24", "v25", "v26", "v27", "v28", "v30", "v32", "v33", "v34",      \
    "v35", "v36", "v38"

struct JRegs {
    float4 x[JB];      // x, y, z relative to the row chunk's centre; m
    float s[JB][4];    // sums of m_i r^-3 (x_j - x_i) and of m_i r^-1
};

// FIRST starts the j sums (saves clearing them).
template <bool FIRST>
__device__ __forceinline__ void sym_group(const float4 &xi, float (&s)[4], JRegs &j)
{
    if (FIRST)
        asm volatile(SYM_GROUP("v_mul_f32_e32")
            : [ax] "+v"(s[0]), [ay] "+v"(s[1]), [az] "+v"(s[2]), [ap] "+v"(s[3]), SYM_J_SUMS("=&v")
            : SYM_INPUTS
            : SYM_TEMPS);
    else
        asm volatile(SYM_GROUP("v_fmac_f32_e32")
            : [ax] "+v"(s[0]), [ay] "+v"(s[1]), [az] "+v"(s[2]), [ap] "+v"(s[3]), SYM_J_SUMS("+v")
            : SYM_INPUTS
            : SYM_TEMPS);
}

template <int NW>
struct SymLds {
    float4 xi[2][TC];               // row chunk, double buffered
    double si[2][NW][4][TC];        // row sums of each wave, double buffered
    float4 xj[NW][JC][TC];          // column chunks relative to the row centre
    double sj[NW][JC][4][TC];       // column sums
};

// One workgroup of NW waves per superblock pair.  The waves own JC column
// chunks each (NW * JC form a column group) and walk the row chunks together;
// per row chunk each wave re-expresses its columns relative to the row's
// centre, evaluates its marked chunk pairs and leaves its row sums in LDS,
// where one wave (in turn) adds the NW sums in order to the item's row slab.
template <int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_sym(SymArgs a)
{
    __shared__ SymLds<NW> lds;
    const int lane = threadIdx.x & 63;
    const int w = uniform_i(threadIdx.x >> 6);
    const int p = lane >> 4, q = lane & 15;
    int bi, bj, item = (int)blockIdx.x;
    if (a.sets) {
        const int2 it = a.items[item];
        a = sym_view(a, it.x);
        item = uniform_i(it.y);
    }
    sym_item(item, a.nsb, bi, bj);
    const int ci0 = bi * a.sb, ci1 = min(ci0 + a.sb, a.nchunks);
    const int cj0 = bj * a.sb, cj1 = min(cj0 + a.sb, a.nchunks);
    const bool diag = bi == bj;
    double *const rows = a.partial + (int64_t)bj * 4 * a.n;
    double *const cols = a.partial + (int64_t)(diag ? a.nsb : bi) * 4 * a.n;
    const double len = a.bbox[6], unit = a.bbox[7];
    unsigned blocks = 0;   // wave-uniform: chunk pairs evaluated
    __builtin_amdgcn_s_setprio(3);

    for (int cg = cj0; cg < cj1; cg += NW * JC) {
        const int cw = cg + w * JC;   // this wave's first column chunk
        double xj[JC], yj[JC], zj[JC];
        float mj[JC];
#pragma unroll
        for (int c = 0; c < JC; ++c) {
            const int64_t j = (int64_t)min(cw + c, a.nchunks - 1) * TC + lane;
            xj[c] = a.p.x[j];
            yj[c] = a.p.y[j];
            zj[c] = a.p.z[j];
            mj[c] = (float)(a.p.m[j] * unit);
#pragma unroll
            for (int k = 0; k < 4; ++k) lds.sj[w][c][k][lane] = 0.0;
        }
        // diagonal items: rows past the column group hold no pair ci < cj
        const int ce = diag && cg > cj0 ? min(ci1, cg + NW * JC) : ci1;
        __syncthreads();   // the previous group is done with lds.xi and lds.si
        for (int ci = ci0 - 1; ci < ce; ++ci) {
            // the wave whose turn it is fetches the next row chunk
            const bool fetch = ci + 1 < ce && ((ci + 1) & (NW - 1)) == w;
            double nx = 0.0, ny = 0.0, nz = 0.0, nm = 0.0;
            double ox = 0.0, oy = 0.0, oz = 0.0;
            if (fetch) {
                const int64_t i = (int64_t)(ci + 1) * TC + lane;
                nx = a.p.x[i];
                ny = a.p.y[i];
                nz = a.p.z[i];
                nm = a.p.m[i];
                chunk_centre(a.chunks + ci + 1, ox, oy, oz);
            }
            double old[4] = {0.0, 0.0, 0.0, 0.0};
            const int64_t irow = (int64_t)ci * TC + lane;
            const bool mine = ci >= ci0 && (ci & (NW - 1)) == w && irow < a.n;
            if (mine && cg > cj0)
                for (int k = 0; k < 4; ++k) old[k] = rows[k * a.n + irow];
            if (ci >= ci0) {
                const int buf = ci & 1;
                unsigned bits = 0;
                if (cw < cj1)
                    bits = (unsigned)(load_scalar(a.sym + (int64_t)ci * a.words + (cw >> 6)) >> (cw & 63)) &
                           0xfu;
                if (cw + JC > cj1) bits &= (1u << max(0, cj1 - cw)) - 1u;
                if (diag) bits &= ci < cw ? 0xfu : (ci - cw >= JC ? 0u : 0xfu & (0xeu << (ci - cw)));
                bits = (unsigned)uniform_i((int)bits);
                float si[IA][4];
                if (bits) {
                    double cx, cy, cz;
                    chunk_centre(a.chunks + ci, cx, cy, cz);
                    wave_lds_sync();
#pragma unroll
                    for (int c = 0; c < JC; ++c)
                        lds.xj[w][c][lane] = make_float4((float)((xj[c] - cx) * len),
                                                         (float)((yj[c] - cy) * len),
                                                         (float)((zj[c] - cz) * len), mj[c]);
                    float4 xi[IA];
#pragma unroll
                    for (int r = 0; r < IA; ++r) {
                        xi[r] = lds.xi[buf][p * IA + r];
#pragma unroll
                        for (int k = 0; k < 4; ++k) si[r][k] = 0.0f;
                    }
                    wave_lds_sync();
                    JRegs j;
                    int c = __builtin_ctz(bits);
#pragma unroll
                    for (int b = 0; b < JB; ++b) j.x[b] = lds.xj[w][c][b * NQ + q];
                    for (unsigned left = bits & (bits - 1);; left &= left - 1) {
                        __builtin_amdgcn_s_setprio(0);
                        sym_group<true>(xi[0], si[0], j);
#pragma unroll
                        for (int r = 1; r < IA; ++r) sym_group<false>(xi[r], si[r], j);
                        __builtin_amdgcn_s_setprio(3);
                        // the next columns are read while these are reduced
                        const int cn = left ? __builtin_ctz(left) : c;
#pragma unroll
                        for (int b = 0; b < JB; ++b) j.x[b] = lds.xj[w][cn][b * NQ + q];
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            const float u = halves32(j.s[0][k], j.s[2][k]);
                            const float v = halves32(j.s[1][k], j.s[3][k]);
                            __hip_atomic_fetch_add(&lds.sj[w][c][k][lane], (double)halves16(u, v),
                                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                        }
                        if (!left) break;
                        c = cn;
                    }
                    blocks += (unsigned)__builtin_popcount(bits);
                    // row sums: over the 16 lanes q, lane q left with row q
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        float u[IA];
#pragma unroll
                        for (int r = 0; r < IA; ++r) u[r] = si[r][k];
                        row_halves8(u);
                        row_halves4(u);
#pragma unroll
                        for (int r = 0; r < 2; ++r)
                            u[r] = quad_step<0x4e>(u[r], u[r + 2], (q & 2) != 0);    // quad 2,3,0,1
                        lds.si[buf][w][k][lane] =
                            (double)quad_step<0xb1>(u[0], u[1], (q & 1) != 0);       // quad 1,0,3,2
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k) lds.si[buf][w][k][lane] = 0.0;
                }
            }
            if (fetch)
                lds.xi[(ci + 1) & 1][lane] = make_float4((float)((nx - ox) * len), (float)((ny - oy) * len),
                                                         (float)((nz - oz) * len), (float)(nm * unit));
            __syncthreads();
            if (mine) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    double s = lds.si[ci & 1][0][k][lane];
#pragma unroll
                    for (int v = 1; v < NW; ++v) s += lds.si[ci & 1][v][k][lane];
                    rows[k * a.n + irow] = old[k] + (k == 3 ? -s : s);
                }
            }
        }
        wave_lds_sync();
#pragma unroll
        for (int c = 0; c < JC; ++c) {
            const int64_t j = (int64_t)(cw + c) * TC + lane;
            if (cw + c < cj1 && j < a.n)
#pragma unroll
                for (int k = 0; k < 4; ++k) cols[k * a.n + j] = -lds.sj[w][c][k][lane];
        }
    }
    if (a.stats && lane == 0 && blocks)
        atomicAdd(&stat_copy(a.stats)[0], 2ull * blocks);   // both orders of each chunk pair
}

// Fixed-order FP64 sum of a particle's slabs and of its row's segments,
// scattered to input order.
__global__ __launch_bounds__(256) void k_sym_reduce(SymArgs a)
{
    int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
    if (a.sets) {   // a block is a tile, of one set
        const int set = a.setof[blockIdx.x * (int64_t)CHUNKS];
        a = sym_view(a, set);
        i -= a.sets[set].pofs;
    }
    if (i >= a.n) return;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int b = 0; b <= a.nsb; ++b) {
        const double *p = a.partial + (int64_t)b * 4 * a.n + i;
        for (int k = 0; k < 4; ++k) s[k] += p[k * a.n];
    }
    // back to the caller's units: a has m / r^2, the potential m / r
    const double len = a.fp64 ? 1.0 : a.bbox[6], unit = a.fp64 ? 1.0 : 1.0 / a.bbox[7];
    // (factor by factor: len^2 alone may leave the range)
    for (int k = 0; k < 3; ++k) s[k] = s[k] * unit * len * len;
    s[3] = s[3] * unit * len;
    const int c = (int)(i / TC), ns = a.psi ? 5 : 4;
    const int e = a.seg[c + 1];
    double psi = 0.0;
    for (int g = a.seg[c]; g < e; ++g) {
        const double *p = a.segsum + (int64_t)g * ns * TC + (i & (TC - 1));
        for (int k = 0; k < 4; ++k) s[k] += p[k * TC];
        if (a.psi) psi += p[4 * TC];
    }
    const int64_t o = a.p.idx[i];
    if (a.psi) {
        const double H = a.p.Hs[i];   // point particles carry no grad-h term
        a.psi[o] = H > 0.0 ? -2.0 * psi / (H * H) : 0.0;
    }
    a.ax[o] = s[0];
    a.ay[o] = s[1];
    a.az[o] = s[2];
    a.pot[o] = s[3];
}

}  // namespace

hipError_t launch_sym_reduce(const SymArgs &a, hipStream_t s)
{
    const int64_t slots = a.sets ? (int64_t)a.nchunks * TC : a.n;
    hipLaunchKernelGGL(k_sym_reduce, dim3((unsigned)((slots + 255) / 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_sym_classify(const SymArgs &a, hipStream_t s)
{
    hipLaunchKernelGGL(k_sym_boxes, dim3((unsigned)((a.nchunks + 255) / 256)), dim3(256), 0, s, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int rows = 4 * CROWS;   // per workgroup
    hipLaunchKernelGGL(k_sym_classify, dim3((unsigned)((a.nchunks + rows - 1) / rows)), dim3(256), 0,
                       s, a);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_sym_segments, dim3(1), dim3(1024), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_sym(const SymArgs &a, hipStream_t s)
{
    const dim3 grid((unsigned)(a.sets ? a.nitems : a.nsb * (a.nsb + 1) / 2));
    switch (a.waves) {
    case 2: hipLaunchKernelGGL((k_sym<2>), grid, dim3(128), 0, s, a); break;
    case 4: hipLaunchKernelGGL((k_sym<4>), grid, dim3(256), 0, s, a); break;
    default: return hipErrorInvalidConfiguration;
    }
    return hipGetLastError();
}

}  // namespace sg
