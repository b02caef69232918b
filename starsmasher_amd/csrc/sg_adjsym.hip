// sg_adjsym.hip -- far pairs of the adjoint (sg_adjoint.hip), each unordered
// pair evaluated once (gfx950).
//
// For a pair of far, Newtonian particles k and l the scalars t, s and
// c = r^-3 (3 t r^-2 - s) of sg_adjoint.hip are the same from both sides, so
// one difference, r^-1, w_k.dr, w_l.dr and c serve both: 40 FP32 VALU
// operations and one v_rsq_f32 against 60 and 2 for the two ordered pairs.
// Chunk pairs, superblock items, slabs and the instruction discipline (joint
// issue of a SIMD's two waves, wave priority around v_rsq_f32, no FMA with
// three sources of one parity) are those of sg_sym.hip; eight values and eight
// sums per particle leave room for 8 rows and 4 columns a lane, an 8 x 8 lane
// grid over 64 rows and 32 columns.
//
// Positions, masses and u are scaled by powers of two (u as the inverse of a
// length, so that all terms of a sum scale alike); the reduce kernel undoes it.
#include "sg_internal.h"
#include "sg_device.h"
#include "sg_lanes.h"

namespace sg {
namespace {

constexpr int RA = 8;          // rows per lane
constexpr int CB = 4;          // columns per lane
constexpr int HC = TC / 2;     // columns per block
constexpr int JC = 2;          // column chunks a wave owns at a time
constexpr int NW = 4;          // waves per workgroup
constexpr int NS = 8;          // sums: G1 (3), G2, G3 (3), GM'
static_assert(RA * 8 == TC && CB * 8 == HC && NW * JC == ADJ_SYM_STEP, "8 x 8 lane grid");

#define ADJ_DIFF(k, dx, dy, dz, r)                                             \
    "v_sub_f32_e32 v" dx ", %[xj" k "], %[xi]\n\t"                             \
    "v_sub_f32_e32 v" dy ", %[yj" k "], %[yi]\n\t"                             \
    "v_sub_f32_e32 v" dz ", %[zj" k "], %[zi]\n\t"                             \
    "v_mul_f32_e32 v" r ", v" dz ", v" dz "\n\t"                               \
    "v_fmac_f32_e32 v" r ", v" dy ", v" dy "\n\t"                              \
    "v_fmac_f32_e32 v" r ", v" dx ", v" dx "\n\t"
#define ADJ_RSQ(ri, r) "v_rsq_f32_e32 v" ri ", v" r "\n\t"
// shared temporaries: even t 40, s 42, r^-3 44; odd wk.dr 41, wl.dr 43, then c
// 45, r^-2 47, r^-3 again 13 (each FMA takes the one whose parity differs)
#define ADJ_SUM(op, k, dx, dy, dz, ri)                                    \
    "v_mul_f32_e32 v47, v" ri ", v" ri "\n\t"                                  \
    "v_mul_f32_e32 v41, %[pi], v" dx "\n\t"                                    \
    "v_mul_f32_e32 v43, %[pj" k "], v" dx "\n\t"                               \
    "v_fmac_f32_e32 v41, %[qi], v" dy "\n\t"                                   \
    "v_fmac_f32_e32 v43, %[qj" k "], v" dy "\n\t"                              \
    "v_fmac_f32_e32 v41, %[si], v" dz "\n\t"                                   \
    "v_fmac_f32_e32 v43, %[sj" k "], v" dz "\n\t"                              \
    "v_mul_f32_e32 v44, v47, v" ri "\n\t"                                      \
    "v_mul_f32_e32 v13, v47, v" ri "\n\t"                                      \
    "v_mul_f32_e32 v40, %[mj" k "], v41\n\t"                                   \
    "v_mul_f32_e32 v42, %[mj" k "], %[ui]\n\t"                                 \
    "v_fma_f32 v40, -%[mi], v43, v40\n\t"                                      \
    "v_fmac_f32_e32 v42, %[mi], %[uj" k "]\n\t"                                \
    "v_mul_f32_e32 v45, %[three], v40\n\t"                                     \
    "v_fmac_f32_e32 %[a0], v13, %[pj" k "]\n\t"                                \
    "v_fmac_f32_e32 %[a1], v44, %[qj" k "]\n\t"                                \
    "v_fma_f32 v45, v45, v47, -v42\n\t"                                        \
    "v_fmac_f32_e32 %[a2], v13, %[sj" k "]\n\t"                                \
    "v_fmac_f32_e32 %[a3], v44, %[mj" k "]\n\t"                                \
    "v_mul_f32_e32 v45, v45, v44\n\t"                                          \
    "v_fmac_f32_e32 %[a7], %[uj" k "], v" ri "\n\t"                            \
    op " %[b0" k "], v13, %[pi]\n\t"                                           \
    op " %[b1" k "], v44, %[qi]\n\t"                                           \
    op " %[b2" k "], v13, %[si]\n\t"                                           \
    op " %[b3" k "], v44, %[mi]\n\t"                                           \
    "v_fmac_f32_e32 %[a7], v44, v43\n\t"                                       \
    op " %[b7" k "], %[ui], v" ri "\n\t"                                       \
    "v_fmac_f32_e32 %[a4], v45, v" dx "\n\t"                                   \
    "v_fmac_f32_e32 %[a5], v45, v" dy "\n\t"                                   \
    "v_fmac_f32_e32 %[a6], v45, v" dz "\n\t"                                   \
    op " %[b4" k "], v45, v" dx "\n\t"                                         \
    op " %[b5" k "], v45, v" dy "\n\t"                                         \
    op " %[b6" k "], v45, v" dz "\n\t"                                         \
    "v_fma_f32 %[b7" k "], -v44, v41, %[b7" k "]\n\t"
#define ADJ_GROUP(op)                                                          \
    ADJ_DIFF("0", "8", "10", "12", "9") ADJ_DIFF("1", "16", "18", "20", "17")  \
    ADJ_DIFF("2", "24", "26", "28", "25") ADJ_DIFF("3", "32", "34", "36", "33") \
    "s_setprio 3\n\t"                                                          \
    ADJ_RSQ("14", "9") ADJ_RSQ("22", "17") ADJ_RSQ("30", "25") ADJ_RSQ("38", "33") \
    "s_setprio 0\n\t"                                                          \
    ADJ_SUM(op, "0", "8", "10", "12", "14")                                \
    ADJ_SUM(op, "1", "16", "18", "20", "22")                               \
    ADJ_SUM(op, "2", "24", "26", "28", "30")                               \
    ADJ_SUM(op, "3", "32", "34", "36", "38")
#define ADJ_J1(c, k)                                                           \
    [b0##k] c(j.s[k][0]), [b1##k] c(j.s[k][1]), [b2##k] c(j.s[k][2]), [b3##k] c(j.s[k][3]), \
    [b4##k] c(j.s[k][4]), [b5##k] c(j.s[k][5]), [b6##k] c(j.s[k][6]), [b7##k] c(j.s[k][7])
#define ADJ_J_SUMS(c) ADJ_J1(c, 0), ADJ_J1(c, 1), ADJ_J1(c, 2), ADJ_J1(c, 3)
#define ADJ_IN1(k)                                                             \
    [xj##k] "v"(j.x[k].x), [yj##k] "v"(j.x[k].y), [zj##k] "v"(j.x[k].z), [mj##k] "v"(j.x[k].w), \
    [pj##k] "v"(j.w[k].x), [qj##k] "v"(j.w[k].y), [sj##k] "v"(j.w[k].z), [uj##k] "v"(j.w[k].w)
#define ADJ_INPUTS                                                             \
    [xi] "v"(x.x), [yi] "v"(x.y), [zi] "v"(x.z), [mi] "v"(x.w), [pi] "v"(w.x), [qi] "v"(w.y), \
    [si] "v"(w.z), [ui] "v"(w.w), [three] "v"(three), ADJ_IN1(0), ADJ_IN1(1), ADJ_IN1(2), ADJ_IN1(3)
#define ADJ_I_SUMS                                                             \
    [a0] "+v"(s[0]), [a1] "+v"(s[1]), [a2] "+v"(s[2]), [a3] "+v"(s[3]), [a4] "+v"(s[4]), \
    [a5] "+v"(s[5]), [a6] "+v"(s[6]), [a7] "+v"(s[7])
#define ADJ_TEMPS                                                              \
    "v8", "v9", "v10", "v12", "v13", "v14", "v16", "v17", "v18", "v20", "v22", "v24", "v25", \
    "v26", "v28", "v30", "v32", "v33", "v34", "v36", "v38", "v40", "v41", "v42", "v43", "v44", \
    "v45", "v47"

struct Cols {
    float4 x[CB], w[CB];   // x, y, z relative to the row chunk's centre, m; wx, wy, wz, u
    float s[CB][NS];
};

// One row against four columns.  FIRST starts the column sums.
template <bool FIRST>
__device__ __forceinline__ void adj_group(const float4 &x, const float4 &w, float (&s)[NS],
                                          float three, Cols &j)
{
    if (FIRST)
        asm volatile(ADJ_GROUP("v_mul_f32_e32")
                     : ADJ_I_SUMS, ADJ_J_SUMS("=&v")
                     : ADJ_INPUTS
                     : ADJ_TEMPS);
    else
        asm volatile(ADJ_GROUP("v_fmac_f32_e32")
                     : ADJ_I_SUMS, ADJ_J_SUMS("+v")
                     : ADJ_INPUTS
                     : ADJ_TEMPS);
}

struct AdjSymLds {
    float4 xi[2][TC], wi[2][TC];      // row chunk, double buffered
    double di[2][4][TC];              // its m, wx, wy, wz
    float si[2][NW][NS][TC];          // row sums of each wave, double buffered
    float4 xj[NW][JC][TC], wj[NW][JC][TC];
    double sj[NW][JC][NS][TC];        // column sums
};

// m G1 - w G2 + G3 and -GM' of one particle, in the scaled units, from its
// sums; sign -1 for columns, whose dr runs the other way.
__device__ __forceinline__ void combine(const double (&g)[NS], double m, double wx, double wy,
                                        double wz, double sign, double (&out)[4])
{
    out[0] = m * g[0] - wx * g[3] + sign * g[4];
    out[1] = m * g[1] - wy * g[3] + sign * g[5];
    out[2] = m * g[2] - wz * g[3] + sign * g[6];
    out[3] = -g[7];
}

__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_adj_sym(AdjSymArgs a)
{
    __shared__ AdjSymLds lds;
    const SymArgs &y = a.y;
    const int lane = threadIdx.x & 63;
    const int w = uniform_i(threadIdx.x >> 6);
    const int p = lane >> 3, q = lane & 7;
    int bi, bj;
    sym_item((int)blockIdx.x, y.nsb, bi, bj);
    const int ci0 = bi * y.sb, ci1 = min(ci0 + y.sb, y.nchunks);
    const int cj0 = bj * y.sb, cj1 = min(cj0 + y.sb, y.nchunks);
    const bool diag = bi == bj;
    double *const rows = y.partial + (int64_t)bj * 4 * y.n;
    double *const cols = y.partial + (int64_t)(diag ? y.nsb : bi) * 4 * y.n;
    const double len = y.bbox[6], unit = y.bbox[7], ulen = 1.0 / len;
    const float three = 3.0f;
    unsigned blocks = 0;   // wave-uniform: chunk pairs evaluated
    __builtin_amdgcn_s_setprio(3);

    for (int cg = cj0; cg < cj1; cg += NW * JC) {
        const int cw = cg + w * JC;   // this wave's first column chunk
#pragma unroll
        for (int c = 0; c < JC; ++c) {
            const int64_t j = (int64_t)min(cw + c, y.nchunks - 1) * TC + lane;
            lds.wj[w][c][lane] = make_float4((float)a.wx[j], (float)a.wy[j], (float)a.wz[j],
                                             (float)(a.u[j] * ulen));
#pragma unroll
            for (int k = 0; k < NS; ++k) lds.sj[w][c][k][lane] = 0.0;
        }
        const int ce = diag && cg > cj0 ? min(ci1, cg + NW * JC) : ci1;
        __syncthreads();   // the previous group is done with the row buffers
        for (int ci = ci0 - 1; ci < ce; ++ci) {
            // the wave whose turn it is fetches the next row chunk
            if (ci + 1 < ce && ((ci + 1) & (NW - 1)) == w) {
                const int64_t i = (int64_t)(ci + 1) * TC + lane;
                double ox, oy, oz;
                chunk_centre(y.chunks + ci + 1, ox, oy, oz);
                const double mi = y.p.m[i] * unit, wx = a.wx[i], wy = a.wy[i], wz = a.wz[i];
                const int nb = (ci + 1) & 1;
                lds.xi[nb][lane] = make_float4((float)((y.p.x[i] - ox) * len),
                                               (float)((y.p.y[i] - oy) * len),
                                               (float)((y.p.z[i] - oz) * len), (float)mi);
                lds.wi[nb][lane] = make_float4((float)wx, (float)wy, (float)wz, (float)(a.u[i] * ulen));
                lds.di[nb][0][lane] = mi;
                lds.di[nb][1][lane] = wx;
                lds.di[nb][2][lane] = wy;
                lds.di[nb][3][lane] = wz;
            }
            const int64_t irow = (int64_t)ci * TC + lane;
            const bool mine = ci >= ci0 && (ci & (NW - 1)) == w && irow < y.n;
            double old[4] = {0.0, 0.0, 0.0, 0.0}, di[4] = {0.0, 0.0, 0.0, 0.0};
            const int buf = ci & 1;
            if (ci >= ci0) {
                unsigned bits = 0;
                if (cw < cj1)
                    bits = (unsigned)(load_scalar(y.sym + (int64_t)ci * y.words + (cw >> 6)) >> (cw & 63)) &
                           0x3u;
                if (cw + JC > cj1) bits &= (1u << max(0, cj1 - cw)) - 1u;
                if (diag) bits &= ci < cw ? 0x3u : (ci - cw >= JC ? 0u : 0x3u & (0x2u << (ci - cw)));
                bits = (unsigned)uniform_i((int)bits);
                if (bits) {
                    double cx, cy, cz;
                    chunk_centre(y.chunks + ci, cx, cy, cz);
                    wave_lds_sync();
#pragma unroll
                    for (int c = 0; c < JC; ++c) {
                        const int64_t j = (int64_t)min(cw + c, y.nchunks - 1) * TC + lane;
                        lds.xj[w][c][lane] = make_float4(
                            (float)((y.p.x[j] - cx) * len), (float)((y.p.y[j] - cy) * len),
                            (float)((y.p.z[j] - cz) * len), (float)(y.p.m[j] * unit));
                    }
                    float4 xi[RA], wi[RA];
                    float si[RA][NS];
#pragma unroll
                    for (int r = 0; r < RA; ++r) {
                        xi[r] = lds.xi[buf][p * RA + r];
                        wi[r] = lds.wi[buf][p * RA + r];
#pragma unroll
                        for (int k = 0; k < NS; ++k) si[r][k] = 0.0f;
                    }
                    wave_lds_sync();
                    Cols j;
                    // blocks of 32 columns: two of each marked chunk
                    int c = __builtin_ctz(bits), h = 0;
                    unsigned left = bits & (bits - 1);
#pragma unroll
                    for (int b = 0; b < CB; ++b) {
                        j.x[b] = lds.xj[w][c][b * 8 + q];
                        j.w[b] = lds.wj[w][c][b * 8 + q];
                    }
                    for (;;) {
                        __builtin_amdgcn_s_setprio(0);
                        adj_group<true>(xi[0], wi[0], si[0], three, j);
#pragma unroll
                        for (int r = 1; r < RA; ++r) adj_group<false>(xi[r], wi[r], si[r], three, j);
                        __builtin_amdgcn_s_setprio(3);
                        // the next columns are read while these are reduced
                        const bool last = h == 1 && left == 0;
                        const int hn = h ^ 1, cn = h == 1 && left ? __builtin_ctz(left) : c;
                        if (h == 1) left &= left - 1;
#pragma unroll
                        for (int b = 0; b < CB; ++b) {
                            j.x[b] = lds.xj[w][cn][hn * HC + b * 8 + q];
                            j.w[b] = lds.wj[w][cn][hn * HC + b * 8 + q];
                        }
                        // over the 8 lanes p: column 8 (lane >> 4) + q stays, in
                        // the lanes with bit 3 clear its sums 0 - 3, else 4 - 7
                        float v[NS];
#pragma unroll
                        for (int k = 0; k < NS; ++k)
                            v[k] = halves16(halves32(j.s[0][k], j.s[2][k]),
                                            halves32(j.s[1][k], j.s[3][k]));
                        row_halves8(v);
                        const int jj = h * HC + (lane >> 4) * 8 + q, k0 = (lane >> 3 & 1) * 4;
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            __hip_atomic_fetch_add(&lds.sj[w][c][k0 + k][jj], (double)v[k],
                                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                        if (last) break;
                        c = cn;
                        h = hn;
                    }
                    blocks += (unsigned)__builtin_popcount(bits);
                    // row sums: over the 8 lanes q, lane q left with row q
#pragma unroll
                    for (int k = 0; k < NS; ++k) {
                        float u[RA];
#pragma unroll
                        for (int r = 0; r < RA; ++r) u[r] = si[r][k];
                        row_halves4(u);
                        u[0] = quad_step<0x4e>(u[0], u[2], (q & 2) != 0);   // quad 2,3,0,1
                        u[1] = quad_step<0x4e>(u[1], u[3], (q & 2) != 0);
                        lds.si[buf][w][k][lane] = quad_step<0xb1>(u[0], u[1], (q & 1) != 0);
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < NS; ++k) lds.si[buf][w][k][lane] = 0.0f;
                }
                if (mine) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        di[k] = lds.di[buf][k][lane];
                        if (cg > cj0) old[k] = rows[k * y.n + irow];
                    }
                }
            }
            __syncthreads();
            if (mine) {
                double g[NS], out[4];
#pragma unroll
                for (int k = 0; k < NS; ++k) {
                    g[k] = (double)lds.si[buf][0][k][lane];
#pragma unroll
                    for (int v = 1; v < NW; ++v) g[k] += (double)lds.si[buf][v][k][lane];
                }
                combine(g, di[0], di[1], di[2], di[3], 1.0, out);
#pragma unroll
                for (int k = 0; k < 4; ++k) rows[k * y.n + irow] = old[k] + out[k];
            }
        }
        wave_lds_sync();
#pragma unroll
        for (int c = 0; c < JC; ++c) {
            const int64_t j = (int64_t)(cw + c) * TC + lane;
            if (cw + c < cj1 && j < y.n) {
                double g[NS], out[4];
#pragma unroll
                for (int k = 0; k < NS; ++k) g[k] = lds.sj[w][c][k][lane];
                combine(g, y.p.m[j] * unit, a.wx[j], a.wy[j], a.wz[j], -1.0, out);
#pragma unroll
                for (int k = 0; k < 4; ++k) cols[k * y.n + j] = out[k];
            }
        }
    }
    if (y.stats && lane == 0 && blocks)
        atomicAdd(&stat_copy(y.stats)[0], 2ull * blocks);   // both orders of each chunk pair
}

// Fixed-order FP64 sum of a particle's slabs and of its row's segments,
// scattered to input order.
__global__ __launch_bounds__(256) void k_adj_sym_reduce(AdjSymArgs a)
{
    const SymArgs &y = a.y;
    const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
    if (i >= y.n) return;
    double s[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int b = 0; b <= y.nsb; ++b) {
        const double *p = y.partial + (int64_t)b * 4 * y.n + i;
        for (int k = 0; k < 4; ++k) s[k] += p[k * y.n];
    }
    // back to the caller's units: positions' gradients m w / r^3, masses' w / r^2
    const double len = y.bbox[6], unit = 1.0 / y.bbox[7];
    // (factor by factor: their product may leave the range)
    for (int k = 0; k < 3; ++k) s[k] = s[k] * unit * len * len * len;
    s[3] = s[3] * len * len;
    const int c = (int)(i / TC);
    const int e = y.seg[c + 1];
    for (int g = y.seg[c]; g < e; ++g) {
        const double *p = y.segsum + (int64_t)g * 5 * TC + (i & (TC - 1));
        for (int k = 0; k < 5; ++k) s[k] += p[k * TC];
    }
    const int64_t o = y.p.idx[i];
    a.gx[o] = s[0];
    a.gy[o] = s[1];
    a.gz[o] = s[2];
    a.gm[o] = s[3];
    a.gH[o] = s[4];
}

}  // namespace

hipError_t launch_adj_sym(const AdjSymArgs &a, hipStream_t s)
{
    if (a.y.sb % (NW * JC) != 0) return hipErrorInvalidConfiguration;
    const dim3 grid((unsigned)(a.y.nsb * (a.y.nsb + 1) / 2));
    hipLaunchKernelGGL(k_adj_sym, grid, dim3(64 * NW), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_adj_sym_reduce(const AdjSymArgs &a, hipStream_t s)
{
    hipLaunchKernelGGL(k_adj_sym_reduce, dim3((unsigned)((a.y.n + 255) / 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace sg
