// kg_internal.h -- shared pieces of libkgstencil.so (not part of the C ABI).
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/kg_stencil.h"

// Slots of the timing ring: one more than the launches it reports, because a
// launch's start may be the stop event of the launch before it.
constexpr int KG_RING_SLOTS = KG_TIMING_RING + 1;

struct kg_ctx {
    int device;
    hipStream_t queue;                // the context's stream; see kg_stream()
    int timing;                       // per-launch timing on/off
    hipEvent_t* ev_start;             // ring of KG_RING_SLOTS start markers
    hipEvent_t* ev_stop;              // and of stop events
    unsigned char* chained;           // slot's start is the previous slot's stop
    bool last_is_stop;                // the stream's last operation is the newest stop event
    bool stopped;                     // the open launch has its stop event on a kernel
    hipError_t launch_err;            // first error of the open launch's kernels
    long long launches;               // launches recorded so far
    long long drained;                // launches already returned by kg_timing_drain
    const char* last_kernel;          // name of the most recent launch
    double* stats;                    // device partials of kg_field_stats
    double* host;                     // pinned, KG_HOST_RESULTS doubles: where a kernel
                                      // leaves a result that the call waits for; or null
    int cus;                          // compute units of the device
    int lds_cu;                       // LDS bytes per compute unit
};

// A few doubles that a kernel writes straight to host memory arrive with the wait for
// the stream; a copy of its own costs a launch, and one into unpinned memory a wait
// more: kg_field_stats of 65536 points takes 33 us with the copy, 23
// without, a Poisson solve of 512 cells 0.95 and 0.79 ms.  The memory is allocated as
// coherent: what a kernel writes to it is there for any kind of wait, an event's included.
constexpr int KG_HOST_RESULTS = 8;

// Bytes of the context's kg_field_stats scratch.
size_t kg_stats_scratch_bytes();
// The kernels of kg_field_stats on stream st, with their partials in
// scratch (kg_stats_scratch_bytes() bytes); the 5 results land in out (device or
// pinned host memory).  No timing, no copy, no synchronisation.
int kg_field_stats_launch(hipStream_t st, int dtype, size_t n, const void* x, int ref_dtype,
                          const void* ref, double* scratch, double* out);
// Waits for the stream and brings n doubles that its kernels left at `from` (host or
// device memory) to `to`.
int kg_bring_results(hipStream_t st, double* to, const double* from, int n, bool from_host);
// Per-device set-up of the Poisson solver's static workspace (kg_init).
int kg_poisson_static_setup(int device);

// Records the most recent error message (thread-local) and returns the code.
int kg_set_error(int code, const char* fmt, ...);

// Wrap a HIP call: on failure record the message and return KG_ERR_HIP.
#define KG_HIP(call)                                                                       \
    do {                                                                                   \
        hipError_t kg_e_ = (call);                                                         \
        if (kg_e_ != hipSuccess)                                                           \
            return kg_set_error(KG_ERR_HIP, "%s failed: %s (%s:%d)", #call,                \
                                hipGetErrorString(kg_e_), __FILE__, __LINE__);             \
    } while (0)

// The context's stream, for work outside kg_launch(): whatever is put on it
// must not count as part of the next launch's duration.
inline hipStream_t kg_stream(kg_ctx* ctx)
{
    ctx->last_is_stop = false;
    return ctx->queue;
}

// Launch bookkeeping used by every entry point: kg_launch_begin() opens the
// next ring slot and settles where its duration starts, kg_launch() starts a
// kernel with the slot's stop event attached (a second kernel of the same
// entry point takes the event over), kg_launch_end() checks the launch and
// records the stop event where no kernel carries it (graphs, plain launches).
//
// Two event records around every kernel cost the stream two barrier packets:
// 11.2 us per launch of an empty kernel back to back against 2.7 without
// timing, 35.6 against 28.1 for a 27.7 us one.  An event attached to the
// kernel's own packet costs 0-1.3 us (4.0 and 28.1 us per launch); attaching
// a start event too makes the runtime add a marker and more host work (14 and
// 32.8 us).  So a launch that queues behind the previous one, still running,
// starts where that one stops (27.56 us reported for the 27.7 us kernel, 3.60
// for the empty one's 3.5), and only a launch on an idle stream, where nothing
// waits for it, records a start marker.  Should the previous launch end between
// kg_launch_begin's look at it and the kernel's dispatch, that gap counts, as a gap
// between a marker and its kernel does.
int kg_launch_begin(kg_ctx* ctx, const char* name);
int kg_launch_end(kg_ctx* ctx);

template <class... P, class... A>
inline void kg_launch(kg_ctx* ctx, void (*kern)(P...), dim3 grid, dim3 block, size_t smem, A... a)
{
    static_assert(sizeof...(P) == sizeof...(A), "one argument per kernel parameter");
    std::tuple<P...> args(static_cast<P>(a)...);
    hipEvent_t stop = ctx->timing ? ctx->ev_stop[ctx->launches % KG_RING_SLOTS] : nullptr;
    std::apply([&](P&... p) {
        void* ptr[] = {(void*)&p...};
        const hipError_t e = hipExtLaunchKernel((const void*)kern, grid, block, ptr, smem, ctx->queue,
                                                nullptr, stop, 0);
        if (e != hipSuccess && ctx->launch_err == hipSuccess) ctx->launch_err = e;
    }, args);
    ctx->stopped = stop != nullptr;
}

// Registry of entry-point name -> kernel symbol, for kg_kernel_regcount.
struct kg_kernel_entry {
    const char* name;
    const void* func;
};
void kg_register_kernel(const char* name, const void* func);

// Device code is loaded lazily, one code object per source file, at the first
// launch of any of its kernels (about 1 ms).  kg_init calls these so that the
// load happens in the init phase, not inside the first timed launch.
int kg_preload_stencil3d();
int kg_preload_tricubic();
int kg_preload_stencil2d();
int kg_preload_matmul();
int kg_preload_util();
int kg_preload_life();
int kg_preload_typed();
int kg_preload_batch();
int kg_preload_poisson();
int kg_preload_vecmath();
int kg_preload_kernel(const void* func);

// Validation helpers shared by the entry points.
int kg_check_ctx(kg_ctx* ctx);
int kg_check_dims3(int nx, int ny, int ns);
int kg_check_dims2(int nx, int ny);
int kg_check_plane_bytes(long long points, int elem_bytes);
// True when every pointer is 16-byte aligned: together with rows of whole
// 16-byte lanes (two doubles, four floats) kernels then take their aligned form,
// otherwise the one for rows of any length and alignment or one point per lane.
template <class... P>
inline bool kg_aligned16(const P*... p)
{
    return !((0u | ... | (unsigned)((uintptr_t)p & 15u)));
}

// Workgroups are dispatched round-robin over the 8 XCDs of an MI355X; each XCD
// has its own L2.  kg_xcd_swizzle maps the hardware workgroup id to a logical
// tile id so that XCD x receives the contiguous logical range
// [x*n/8, (x+1)*n/8): neighbouring tiles (which share halo cache lines) then
// sit in the same L2.  Ids past the last multiple of 8 map to themselves.
#ifndef KG_XCD_SWIZZLE
#define KG_XCD_SWIZZLE 1
#endif
__device__ __forceinline__ unsigned kg_xcd_swizzle(unsigned b, unsigned n)
{
    if (!KG_XCD_SWIZZLE) return b;
    const unsigned per = n >> 3;
    if (b < (per << 3)) return (b & 7u) * per + (b >> 3);
    return b;
}

#define KG_NUM_XCD 8

// Dynamic LDS to reserve (unused) so that at most occ workgroups, each with
// static_lds bytes of its own, are resident on one compute unit: occ+1
// workgroups of lds_cu/occ - 256 bytes do not fit in lds_cu.  0 when occ <= 0
// or the workgroup's own LDS already allows no more.
inline size_t kg_occupancy_lds(const kg_ctx* ctx, int occ, size_t static_lds)
{
    if (occ <= 0) return 0;
    const size_t per = (size_t)ctx->lds_cu / (size_t)occ;
    return per > static_lds + 256 ? per - static_lds - 256 : 0;
}

// Planes each workgroup marches when its launch covers nz of them with
// `tiles` tiles side by side: kc on large grids; on small ones, where the kc of a
// full chip would leave compute units idle or a last round nearly empty, the
// number below kc that takes the least time.  A workgroup takes about kc + fill
// planes' time (fill: the planes it loads before the first result) and the
// device runs per_cu workgroups per compute unit at once.
// Whole chunks against these: 64x32x32 lapgsrb 30 -> 5.7 us, wave13pt 20 -> 5.6,
// tricubic 20 -> 6.2; 128^3 lapgsrb 35 -> 12.7, wave13pt 22 -> 11.2, its FP32 form
// 55 -> 10.6 and BF16 72 -> 13.1; 200^3 wave13pt 54 -> 43.5, FP32 55 -> 19.9, BF16
// 72 -> 26.  From four rounds of workgroups on the chunk of the large grids is
// kept: there the last round is a small part and longer chunks read less.
inline int kg_fit_chunk(const kg_ctx* ctx, long long tiles, int nz, int kc, int per_cu, int fill)
{
    const long long room = (long long)per_cu * ctx->cus;
    if (tiles <= 0 || nz <= 0 || tiles * ((nz + kc - 1) / kc) >= 4 * room) return kc;
    auto time = [&](int k) {
        const long long wgs = tiles * ((nz + k - 1) / k);
        return (wgs + room - 1) / room * (std::min(k, nz) + fill);
    };
    int best = kc;
    for (int k = std::min(kc, nz); k >= 1; k--)
        if (time(k) < time(best)) best = k;
    // the planes two chunks share are read twice: a small gain is none
    return time(best) * 100 < time(kc) * 85 ? best : kc;
}

// kg_xcd_chunk deals runs of `chunk` consecutive logical tiles to the XCDs in
// turn: XCD x receives logical chunks x, x+8, x+16, ..., so at any moment
// the 8 XCDs work on 8 consecutive chunks (the chip streams one window) and
// the tiles of a chunk share one L2.  Ids past the last whole round of 8
// chunks map to themselves.
__device__ __forceinline__ unsigned kg_xcd_chunk(unsigned b, unsigned n, unsigned chunk)
{
    if (!KG_XCD_SWIZZLE) return b;
    const unsigned round = chunk * KG_NUM_XCD;
    if (b >= n / round * round) return b;
    const unsigned x = b % KG_NUM_XCD, s = b / KG_NUM_XCD;   // XCD, its sequence number
    return ((s / chunk) * KG_NUM_XCD + x) * chunk + s % chunk;
}

// Logical tile id of workgroup b of n, for tiles numbered x fastest with ntx
// tiles per tile row.  ORD 0: hardware order (consecutive tiles on different
// XCDs; the chip streams one window).  ORD 1: each XCD takes a contiguous
// eighth (kg_xcd_swizzle).  ORD >= 2: chunks of ORD tile rows per XCD
// (kg_xcd_chunk): a tile's x-neighbours and most of its y-neighbours share
// its L2, and the chip still streams one window of 8 * ORD tile rows.
template <int ORD>
__device__ __forceinline__ unsigned kg_tile_order(unsigned b, unsigned n, unsigned ntx)
{
    static_assert(ORD >= 0, "tile order");
    if constexpr (ORD == 0) return b;
    else if constexpr (ORD == 1) return kg_xcd_swizzle(b, n);
    else return kg_xcd_chunk(b, n, ntx * (unsigned)ORD);
}

// f(std::integral_constant<int, 0>{}), ..., f(std::integral_constant<int, N-1>{}):
// a loop unrolled at compile time with the index usable as a constant.
template <class Fn, int... I>
__device__ __forceinline__ void kg_static_for_impl(Fn&& f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class Fn>
__device__ __forceinline__ void kg_static_for(Fn&& f)
{
    kg_static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// Streaming store for stencil outputs.  Output grids are written once per step
// and not read again by the same kernel; marking the store non-temporal keeps
// it from displacing, in L2, the input lines that neighbouring rows and planes
// are about to re-read.  Measured on MI355X (512x256x256 laplacian): 153 us
// with ordinary stores, 87 us with non-temporal ones.
template <typename T>
__device__ __forceinline__ void kg_st(T* p, T v)
{
    __builtin_nontemporal_store(v, p);
}
