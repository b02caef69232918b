// A device made of bookkeeping, to run the host code of sg_capi.cpp without a
// GPU: allocations come from a budget and hold nothing, copies to the host give
// zeros, launches succeed and are checked for the buffers they would work in.
// Built and driven by tests/test_allocation.py.
#include <hip/hip_runtime.h>

#include "sphgrav.h"
#include "sg_internal.h"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {

std::map<char *, size_t> live;
size_t used = 0, budget = ~(size_t)0;
char *next_address = (char *)0x100000000000;
int mallocs = 0, frees = 0, graphs = 0, fail_at = 0;
std::string ran;     // names of the pair passes launched
std::string fault;   // the first launch that would leave its buffers

// Whether [p, p + bytes) lies in one live allocation.
void need(const char *what, const void *p, size_t bytes)
{
    auto it = live.upper_bound((char *)p);
    if (it != live.begin() && (--it, (char *)p >= it->first) &&
        (char *)p + bytes <= it->first + it->second)
        return;
    if (fault.empty()) fault = std::string(what) + " " + std::to_string(bytes) + " bytes";
}

void set(const sg::SortedSet &s)
{
    for (const double *p : {s.x, s.y, s.z, s.m, s.Hs}) need("sorted set", p, 8 * s.padded);
    need("sorted index", s.idx, 4 * s.padded);
}

void prep(const sg::PrepBuffers &b, int64_t n)
{
    need("keys_in", b.keys_in, 8 * n);
    need("keys_out", b.keys_out, 8 * n);
    need("vals_in", b.vals_in, 4 * n);
    need("vals_out", b.vals_out, 4 * n);
    need("bbox", b.bbox, 64);
    need("err", b.err, 4);
}

void unordered(const char *name, const sg::SymArgs &a, int sums)
{
    ran += std::string(name) + " ";
    need("boxes", a.boxes, (size_t)a.nchunks * 32);
    need("segments", a.seg, ((size_t)a.nchunks + 3) * 4);
    need("segment sums", a.segsum, ((size_t)sg::SYM_SEGS + a.nchunks) * sums * sg::TC * 8);
    if (!a.sets) {
        set(a.p);
        need("bits", a.sym, (size_t)a.nchunks * a.words * 8);
        need("slabs", a.partial, (size_t)(a.nsb + 1) * 4 * a.n * 8);
    } else {
        need("items", a.items, (size_t)a.nitems * 8);
        need("set of each chunk", a.setof, (size_t)a.nchunks * 4);
    }
}

}  // namespace

extern "C" {

void fake_reset(long long bytes, int fail)   // fail: the malloc of that number fails
{
    budget = bytes < 0 ? ~(size_t)0 : (size_t)bytes;
    mallocs = frees = graphs = 0;
    fail_at = fail;
    ran.clear();
    fault.clear();
}
int fake_mallocs(void) { return mallocs; }
int fake_frees(void) { return frees; }
int fake_graphs(void) { return graphs; }
long long fake_used(void) { return (long long)used; }
const char *fake_ran(void) { return ran.c_str(); }
const char *fake_fault(void) { return fault.c_str(); }

hipError_t hipMalloc(void **p, size_t n)
{
    ++mallocs;
    *p = nullptr;
    if (mallocs == fail_at || n > budget - used || used > budget) return hipErrorOutOfMemory;
    *p = next_address;
    live[next_address] = n;
    next_address += (n + 4095) / 4096 * 4096 + 4096;
    used += n;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    ++frees;
    auto it = live.find((char *)p);
    if (it == live.end()) return hipErrorInvalidValue;
    used -= it->second;
    live.erase(it);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *free, size_t *total)
{
    *total = (size_t)288 << 30;
    *free = budget == ~(size_t)0 ? *total : (used < budget ? budget - used : 0);
    return hipSuccess;
}
hipError_t hipMemcpy(void *dst, const void *src, size_t n, hipMemcpyKind kind)
{
    if (kind == hipMemcpyDeviceToHost) {
        need("copy to the host", src, n);
        std::memset(dst, 0, n);
    } else {
        need("copy to the device", dst, n);
    }
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind kind, hipStream_t)
{
    return hipMemcpy(dst, src, n, kind);
}
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)8; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)8; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)8; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { ++graphs; *g = (hipGraph_t)8; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *g, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    *g = (hipGraphExec_t)8;
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }

}  // extern "C"

namespace sg {

hipError_t launch_validate_bbox(const double *, const double *, const double *, const double *,
                                const double *, int n, PrepBuffers &b, hipStream_t)
{
    prep(b, n);
    return hipSuccess;
}
hipError_t launch_morton(const double *, const double *, const double *, int, int n,
                         const PrepBuffers &b, hipStream_t)
{
    prep(b, n);
    return hipSuccess;
}
hipError_t launch_morton_batch(const double *, const double *, const double *, int n,
                               const int64_t *, int, const PrepBuffers &b, hipStream_t)
{
    prep(b, n);
    return hipSuccess;
}
hipError_t sort_pairs_temp_bytes(int n, size_t *bytes) { *bytes = (size_t)n * 4; return hipSuccess; }
hipError_t sort_pairs(void *tmp, size_t bytes, const uint64_t *, uint64_t *, const int *, int *,
                      int n, hipStream_t)
{
    need("sort storage", tmp, (size_t)n * 4);
    return bytes >= (size_t)n * 4 ? hipSuccess : hipErrorInvalidValue;
}
hipError_t merge_sort_pairs(void *, size_t, const uint64_t *, uint64_t *, const int *, int *, int,
                            hipStream_t)
{
    return hipSuccess;
}
hipError_t launch_gather(const double *, const double *, const double *, const double *,
                         const double *, const int *, int, int64_t padded, double *ox, double *oy,
                         double *oz, double *om, double *oH, int *oidx, hipStream_t)
{
    for (double *p : {ox, oy, oz, om, oH}) need("i set", p, 8 * padded);
    need("i index", oidx, 4 * padded);
    return hipSuccess;
}
hipError_t launch_gather_batch(const double *, const double *, const double *, const double *,
                               const double *, const int *, const int64_t *, const BatchSet *, int,
                               int64_t padded, double *ox, double *oy, double *oz, double *om,
                               double *oH, int *oidx, hipStream_t)
{
    for (double *p : {ox, oy, oz, om, oH}) need("batch set", p, 8 * padded);
    need("batch index", oidx, 4 * padded);
    return hipSuccess;
}
hipError_t launch_gather_cot(const double *, const double *, const double *, const double *,
                             const int *, int, int64_t padded, double *a, double *b, double *c,
                             double *d, const PrepBuffers &, hipStream_t)
{
    for (double *p : {a, b, c, d}) need("cotangents", p, 8 * padded);
    return hipSuccess;
}
hipError_t launch_prep_small(const double *, const double *, const double *, const double *,
                             const double *, int n, const PrepBuffers &b, unsigned long long *,
                             hipStream_t)
{
    prep(b, n);
    return hipSuccess;
}
hipError_t launch_gather_tiles(const double *, const double *, const double *, const double *,
                               const double *, int n, int64_t padded, const PrepBuffers &b,
                               hipStream_t)
{
    prep(b, n);
    set(SortedSet{b.sx, b.sy, b.sz, b.sm, b.sH, b.sidx, n, padded});
    need("tiles", b.tiles, (size_t)(padded / TJ) * sizeof(TileMeta));
    need("chunks", b.chunks, (size_t)(padded / TC) * sizeof(TileMeta));
    return hipSuccess;
}
hipError_t launch_tile_meta(const double *, const double *, const double *, const double *,
                            int ntiles, TileMeta *tiles, TileMeta *chunks, hipStream_t)
{
    need("tiles", tiles, (size_t)ntiles * sizeof(TileMeta));
    need("chunks", chunks, (size_t)ntiles * CHUNKS * sizeof(TileMeta));
    return hipSuccess;
}
hipError_t launch_fill_zero_int(int *p, int n, hipStream_t) { need("fill", p, 4 * (size_t)n); return hipSuccess; }
hipError_t launch_potential_energy(const double *, const double *, int, double *, int, hipStream_t)
{
    return hipSuccess;
}
hipError_t launch_pair_far(int, const PairArgs &a, int, hipStream_t)
{
    ran += a.wave ? "wave " : "ordered ";
    set(a.j);
    need("partial sums", a.partial, (size_t)a.jsplit * 4 * a.ni * 8);
    if (a.psi) need("psi partial sums", a.psipart, (size_t)a.jsplit * a.ni * 8);
    return hipSuccess;
}
hipError_t launch_pair_near(int, const PairArgs &, hipStream_t) { return hipSuccess; }
hipError_t launch_reduce_partials(const PairArgs &, hipStream_t) { return hipSuccess; }
hipError_t launch_psi_only(const PairArgs &a, hipStream_t)
{
    set(a.j);
    need("psi partial sums", a.psipart, (size_t)a.jsplit * a.ni * 8);
    return hipSuccess;
}
hipError_t launch_batch(int, const BatchArgs &a, int, int, int, hipStream_t)
{
    ran += "ordered_batch ";
    need("work items", a.items, (size_t)a.nitems * 8);
    need("queue", a.counter, 4);
    return hipSuccess;
}
bool pair_config_supported(int, int, int) { return true; }
bool batch_config_supported(int, int) { return true; }
int batch_resident_workgroups(int, int, int, int, int) { return 1024; }
hipError_t launch_set_boxes(const SymArgs &, int nsets, double *boxes, hipStream_t)
{
    need("boxes of the sets", boxes, (size_t)nsets * 64);
    return hipSuccess;
}
hipError_t launch_sym_classify(const SymArgs &, hipStream_t) { return hipSuccess; }
hipError_t launch_sym(const SymArgs &a, hipStream_t) { unordered("sym", a, a.psi ? 5 : 4); return hipSuccess; }
hipError_t launch_sym64(const SymArgs &a, hipStream_t) { unordered("sym64", a, a.psi ? 5 : 4); return hipSuccess; }
hipError_t launch_sym_rest(const SymArgs &, hipStream_t) { return hipSuccess; }
hipError_t launch_sym_reduce(const SymArgs &, hipStream_t) { return hipSuccess; }
hipError_t launch_adj_sym(const AdjSymArgs &a, hipStream_t) { unordered("adj_sym", a.y, 5); return hipSuccess; }
hipError_t launch_adj_sym_rest(const AdjSymArgs &, hipStream_t) { return hipSuccess; }
hipError_t launch_adj_sym_reduce(const AdjSymArgs &, hipStream_t) { return hipSuccess; }
hipError_t launch_adj_far(int, const AdjArgs &a, int wg, hipStream_t)
{
    ran += "adj_ordered" + std::to_string(wg) + " ";
    need("gradient partial sums", a.partial, (size_t)a.jsplit * 5 * a.n * 8);
    need("near flags", a.nearflag, (size_t)a.ngroups * a.ntiles);
    return hipSuccess;
}
hipError_t launch_adj_wave(const AdjArgs &a, hipStream_t)
{
    ran += "adj_wave ";
    need("gradient partial sums", a.partial, (size_t)a.jsplit * 5 * a.n * 8);
    return hipSuccess;
}
hipError_t launch_adj_near(int, const AdjArgs &, hipStream_t) { return hipSuccess; }
hipError_t launch_adj_reduce(const AdjArgs &, hipStream_t) { return hipSuccess; }
bool adj_config_supported(int wg) { return wg == 64 || wg == 128 || wg == 256; }

}  // namespace sg
