// sg_sym64.hip -- far pairs of a whole FP64 set, each unordered pair evaluated
// once (gfx950).
//
// One difference, r^2 and reciprocal square root serve both particles: 24 FP64
// operations and one v_rsq_f64 per unordered pair against 34 and 2 for the two
// ordered ones.  Chunk pairs, superblock items and slabs are those of
// sg_sym.hip.  FP64 instructions of a SIMD's waves never issue together, so
// there is nothing to pair up and the body is plain code; what bounds it is
// their number.  A lane of the 8 x 8 grid holds 4 columns and their sums and
// the sums of 8 rows in registers and reads the rows from LDS, one at a time
// (its eight lanes read one address).
//
// At 131,072 particles 27 VALU instructions per unordered pair (24 of the pair,
// the rest in the reductions over the lanes) keep the vector units busy for 92%
// of the 7.9 ms, at three waves per SIMD; the ordered kernel took 12.2 ms.
//
// Differences are taken between the positions as given, one rounding each.
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
static_assert(RA * 8 == TC && CB * 8 == HC && NW * JC == SYM64_STEP, "8 x 8 lane grid");

// lane l's value of the lane that the DPP control names
template <int CTRL>
__device__ __forceinline__ double dpp64(double v)
{
    int w[2];
    __builtin_memcpy(w, &v, 8);
    w[0] = __builtin_amdgcn_update_dpp(0, w[0], CTRL, 0xf, 0xf, true);
    w[1] = __builtin_amdgcn_update_dpp(0, w[1], CTRL, 0xf, 0xf, true);
    __builtin_memcpy(&v, w, 8);
    return v;
}
// One step of a reduce-scatter: the lanes with `upper` unset keep a, the others
// b, and both add the partner lane's.
template <int CTRL>
__device__ __forceinline__ double step64(double a, double b, bool upper)
{
    const double keep = upper ? b : a, send = upper ? a : b;
    return keep + dpp64<CTRL>(send);
}
// The same over the register halves (lanes from 32, odd rows of 16 lanes).
template <int W>
__device__ __forceinline__ double swap64(double a, double b)
{
    unsigned u[2], v[2];
    __builtin_memcpy(u, &a, 8);
    __builtin_memcpy(v, &b, 8);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const auto r = W == 32 ? __builtin_amdgcn_permlane32_swap(u[k], v[k], false, false)
                               : __builtin_amdgcn_permlane16_swap(u[k], v[k], false, false);
        const unsigned lo = r[0], hi = r[1];
        u[k] = lo;
        v[k] = hi;
    }
    __builtin_memcpy(&a, u, 8);
    __builtin_memcpy(&b, v, 8);
    return a + b;
}

struct Cols64 {
    double x[CB], y[CB], z[CB], m[CB];
    double s[CB][4];
};

struct Sym64Lds {
    double2 xi[2][2][TC];           // row chunk: {x, y}, {z, m}; double buffered
    double si[2][NW][4][TC];        // row sums of each wave, double buffered
    double2 xj[NW][JC][2][TC];      // column chunks
    double sj[NW][JC][4][TC];       // column sums
};

__device__ __forceinline__ void load_cols(Cols64 &j, const double2 (&x)[2][TC], int j0)
{
#pragma unroll
    for (int b = 0; b < CB; ++b) {
        const double2 u = x[0][j0 + b * 8], v = x[1][j0 + b * 8];
        j.x[b] = u.x;
        j.y[b] = u.y;
        j.z[b] = v.x;
        j.m[b] = v.y;
    }
}

// One row against the lane's columns.
__device__ __forceinline__ void row64(const double2 &u, const double2 &v, double (&s)[4], Cols64 &j)
{
#pragma unroll
    for (int b = 0; b < CB; ++b) {
        const double dx = j.x[b] - u.x, dy = j.y[b] - u.y, dz = j.z[b] - v.x;
        const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
        const double ri = rsqrt_pos64(r2);   // far: r^2 >= max(H_i^2, H_j^2) > 0
        const double r3 = ri * ri * ri;
        const double gi = j.m[b] * r3, gj = v.y * r3;
        s[0] = fma(gi, dx, s[0]);
        s[1] = fma(gi, dy, s[1]);
        s[2] = fma(gi, dz, s[2]);
        s[3] = fma(j.m[b], ri, s[3]);
        j.s[b][0] = fma(gj, dx, j.s[b][0]);
        j.s[b][1] = fma(gj, dy, j.s[b][1]);
        j.s[b][2] = fma(gj, dz, j.s[b][2]);
        j.s[b][3] = fma(v.y, ri, j.s[b][3]);
    }
}

__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(3, 3)))
void k_sym64(SymArgs a)
{
    __shared__ Sym64Lds lds;
    const int lane = threadIdx.x & 63;
    const int w = uniform_i(threadIdx.x >> 6);
    const int p = lane >> 3, q = lane & 7;
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
    unsigned blocks = 0;   // wave-uniform: chunk pairs evaluated

    for (int cg = cj0; cg < cj1; cg += NW * JC) {
        const int cw = cg + w * JC;   // this wave's first column chunk
#pragma unroll
        for (int c = 0; c < JC; ++c) {
            const int64_t j = (int64_t)min(cw + c, a.nchunks - 1) * TC + lane;
            lds.xj[w][c][0][lane] = make_double2(a.p.x[j], a.p.y[j]);
            lds.xj[w][c][1][lane] = make_double2(a.p.z[j], a.p.m[j]);
#pragma unroll
            for (int k = 0; k < 4; ++k) lds.sj[w][c][k][lane] = 0.0;
        }
        // diagonal items: rows past the column group hold no pair ci < cj
        const int ce = diag && cg > cj0 ? min(ci1, cg + NW * JC) : ci1;
        __syncthreads();   // the previous group is done with the row buffers
        for (int ci = ci0 - 1; ci < ce; ++ci) {
            // the wave whose turn it is fetches the next row chunk
            if (ci + 1 < ce && ((ci + 1) & (NW - 1)) == w) {
                const int64_t i = (int64_t)(ci + 1) * TC + lane;
                const int nb = (ci + 1) & 1;
                lds.xi[nb][0][lane] = make_double2(a.p.x[i], a.p.y[i]);
                lds.xi[nb][1][lane] = make_double2(a.p.z[i], a.p.m[i]);
            }
            const int64_t irow = (int64_t)ci * TC + lane;
            const bool mine = ci >= ci0 && (ci & (NW - 1)) == w && irow < a.n;
            double old[4] = {0.0, 0.0, 0.0, 0.0};
            const int buf = ci & 1;
            if (ci >= ci0) {
                unsigned bits = 0;
                if (cw < cj1)
                    bits = (unsigned)(a.sym[(int64_t)ci * a.words + (cw >> 6)] >> (cw & 63)) & 0x3u;
                if (cw + JC > cj1) bits &= (1u << max(0, cj1 - cw)) - 1u;
                if (diag) bits &= ci < cw ? 0x3u : (ci - cw >= JC ? 0u : 0x3u & (0x2u << (ci - cw)));
                bits = (unsigned)uniform_i((int)bits);
                if (bits) {
                    double s[RA][4];
#pragma unroll
                    for (int r = 0; r < RA; ++r)
#pragma unroll
                        for (int k = 0; k < 4; ++k) s[r][k] = 0.0;
                    wave_lds_sync();
                    Cols64 j;
                    // blocks of 32 columns: two of each marked chunk
                    int c = __builtin_ctz(bits), h = 0;
                    unsigned left = bits & (bits - 1);
                    load_cols(j, lds.xj[w][c], q);
                    for (;;) {
#pragma unroll
                        for (int b = 0; b < CB; ++b)
#pragma unroll
                            for (int k = 0; k < 4; ++k) j.s[b][k] = 0.0;
#pragma unroll
                        for (int r = 0; r < RA; ++r)
                            row64(lds.xi[buf][0][r * 8 + p], lds.xi[buf][1][r * 8 + p], s[r], j);
                        // the next columns are read while these are reduced
                        const bool last = h == 1 && left == 0;
                        const int hn = h ^ 1, cn = h == 1 && left ? __builtin_ctz(left) : c;
                        if (h == 1) left &= left - 1;
                        load_cols(j, lds.xj[w][cn], hn * HC + q);
                        // over the 8 lanes p: column 8 (lane >> 4) + q stays, in
                        // the lanes with bit 3 clear its sums 0 and 1, else 2 and 3
                        double v[4];
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            v[k] = swap64<16>(swap64<32>(j.s[0][k], j.s[2][k]),
                                              swap64<32>(j.s[1][k], j.s[3][k]));
                        const bool up8 = (lane & 8) != 0;
                        const int jj = h * HC + (lane >> 4) * 8 + q, k0 = up8 ? 2 : 0;
#pragma unroll
                        for (int k = 0; k < 2; ++k)   // row_ror:8
                            __hip_atomic_fetch_add(&lds.sj[w][c][k0 + k][jj],
                                                   step64<0x128>(v[k], v[k + 2], up8),
                                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                        if (last) break;
                        c = cn;
                        h = hn;
                    }
                    blocks += (unsigned)__builtin_popcount(bits);
                    // row sums over the 8 lanes q: of row 8 r + p, r = the bits
                    // (q & 4, q & 2, q & 1), stays
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        double u[RA / 2];
#pragma unroll
                        for (int r = 0; r < RA / 2; ++r)   // row_half_mirror
                            u[r] = step64<0x141>(s[r][k], s[r + 4][k], (q & 4) != 0);
                        u[0] = step64<0x4e>(u[0], u[2], (q & 2) != 0);   // quad 2,3,0,1
                        u[1] = step64<0x4e>(u[1], u[3], (q & 2) != 0);
                        lds.si[buf][w][k][q * 8 + p] = step64<0xb1>(u[0], u[1], (q & 1) != 0);
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k) lds.si[buf][w][k][lane] = 0.0;
                }
                if (mine && cg > cj0)
#pragma unroll
                    for (int k = 0; k < 4; ++k) old[k] = rows[k * a.n + irow];
            }
            __syncthreads();
            if (mine) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    double t = lds.si[buf][0][k][lane];
#pragma unroll
                    for (int v = 1; v < NW; ++v) t += lds.si[buf][v][k][lane];
                    rows[k * a.n + irow] = old[k] + (k == 3 ? -t : t);
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

}  // namespace

hipError_t launch_sym64(const SymArgs &a, hipStream_t s)
{
    if (!a.sets && a.sb % (NW * JC) != 0) return hipErrorInvalidConfiguration;
    const dim3 grid((unsigned)(a.sets ? a.nitems : a.nsb * (a.nsb + 1) / 2));
    hipLaunchKernelGGL(k_sym64, grid, dim3(64 * NW), 0, s, a);
    return hipGetLastError();
}

}  // namespace sg
