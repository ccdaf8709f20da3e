// kg_poisson.hip -- 2D Poisson solve with FP32 multigrid sweeps inside an FP64
// defect-correction loop.
//
// Problem: A u = f on the unit square with u = 0 on the boundary, on an
// (n+1) x (n+1) vertex grid (n cells per side, n a power of two, h = 1/n),
// x fastest.  A is the 9-point operator whose Jacobi sweep is the reference's
// jacobi kernel (jacobi/jacobi.F90:65-67: c0*w + c1*(4 axis neighbours) +
// c2*(4 diagonal neighbours)) plus a right-hand-side term:
//
//   (A u)(i,j) = (20 u - 4 (u_E + u_W + u_N + u_S) - (u_NE + u_NW + u_SE + u_SW)) / (6 h^2)
//
// damped Jacobi: u' = (1-w) u + (w/5) sum_axis + (w/20) sum_diag + (3 w h^2 / 10) f.
//
// Outer loop (FP64): r = f - A u (one pass that also writes r in FP32 as the
// inner right-hand side and sums r^2); stop when ||r||_2 / ||f||_2 < tol; else
// solve A e = r approximately in FP32 (V-cycles: full-weighting restriction,
// bilinear prolongation, damped-Jacobi smoothing, rediscretised coarse
// operators down to 3 x 3 vertices) and set u += e.  The FP32 inner solve
// needs only a few digits per correction; FP64 residuals recover the rest.
//
// The FP32 levels are stored with rows padded to P = N rounded up to 16
// floats, so that their passes work on 16-byte pieces and write whole rows
// (0 at the boundary and padding points): no cache line is written in part.
#include "kg_plane.h"

#include <chrono>
#include <cmath>
#include <mutex>

namespace {

// Tile orders (kg_tile_order).  In the marching passes each XCD takes a contiguous
// eighth of the tile rows (1): tile rows that share rows then follow each other on
// one XCD, although their rows overflow its L2 (pj_up_k reads 1.4 times its input past
// L2).  8192^2: pj_up_k 186 us, pj_down_k 182 and, from 0, 117; in chunks of 2 tile
// rows per XCD 204, 187 and 131, in hardware order 204, 189 and 133.  The FP64 residual
// takes chunks of 2 (259 us; contiguous eighths 272, chunks of 4 or 8 257-263).
#ifndef KG_ORD_PJ
#define KG_ORD_PJ 1
#endif
#ifndef KG_ORD_PJR
#define KG_ORD_PJR 2
#endif

typedef float f2 __attribute__((ext_vector_type(2)));
typedef double d2 __attribute__((ext_vector_type(2)));
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));   // at any element

// ------------------------------------------------------------ a level's passes
// A V-cycle visits a level twice: on the way down two damped Jacobi sweeps, the
// residual and its full-weighting restriction, on the way up the bilinear
// correction and two sweeps.  Each visit is one pass over the level (pj_down_k,
// pj_up_k): a wave takes 64 V columns, V per lane, and marches them along y; an
// incoming row enters a window of three rows, which gives the first sweep of the
// row before it, three of those give the second sweep of the row before that,
// and so on, so that HBM sees u, f and the result once per visit.  The columns
// beside a lane's V come from the neighbouring lanes by DPP.  Every stage makes
// the wave's outermost column on either side invalid; the outer lanes hold only
// such overlap (pieces start every 240 or 112 columns, 64-byte aligned).  Expressions and
// orders are those of separate sweeps, residual and restriction, and so is the
// result, bit for bit.
//
// Bound by HBM on the finest levels: u, f, u' and a quarter of it on the next
// level are 871 MB at 8192^2, 186 us (4.7 TB/s; the best copy reaches 6.3) for
// pj_up_k and 182 for pj_down_k.  Sweep pairs, residual and restriction,
// prolongation and the addition to u as passes of their own took 14.2 of the 17.7 ms
// of an 8192^2 solve (7.5, 3.3, 1.9, 1.5); it takes 9.7 so.  Rows of 64-byte
// multiples and pieces of 240 columns, so that no wave writes part of a sector:
// 5 % faster at 8192^2 than 248 columns of 4-float pitches.  The 4 waves of a
// workgroup lie side by side; one above the other costs 2 % more.  Small levels
// are bound by a wave's march (6 us at 512 cells and below), whose steps V = 2 halves:
// solves of 256 to 1024 cells 0.59, 0.80, 1.01 -> 0.56, 0.76, 0.96 ms.  It is taken where
// 4 rows per wave leave a CU less than 8 waves; elsewhere V = 4 marches less overlap.
constexpr int MW = 4;                  // waves per workgroup, side by side in x
// columns a wave completes, V per lane: 1 or 2 lanes on either side are overlap
template <int V> constexpr int edge_lanes() { return 4 / V; }
template <int V> constexpr int piece() { return V == 4 ? 240 : 112; }

struct Coef {
    float c0, c1, c2, cf;              // sweep: c0 u + c1 axis + c2 diag + cf f
    float inv6h2;
};

// A lane's columns of a row and the ones on either side of them.
template <int V>
struct Row {
    float v[V], l, r;
    __device__ __forceinline__ float at(int i) const { return i < 0 ? l : i > V - 1 ? r : v[i]; }
    __device__ __forceinline__ void sides()
    {
        l = kgp::dpp_shift<kgp::KG_DPP_WAVE_SHR1>(0.f, v[V - 1]);
        r = kgp::dpp_shift<kgp::KG_DPP_WAVE_SHL1>(0.f, v[0]);
    }
};

// damped Jacobi sweep of row b (a below, c above it): u' = c0 u + c1 (W + S + E +
// N) + c2 (SW + NW + SE + NE) + cf f on the interior, 0 elsewhere
template <int V>
__device__ __forceinline__ void pj_sweep(const Coef& k, const Row<V>& a, const Row<V>& b, const Row<V>& c,
                                         const float (&f)[V], bool row_in, const bool (&in)[V], Row<V>& o)
{
#pragma unroll
    for (int v = 0; v < V; v++) {
        const float val = k.c0 * b.v[v] + k.c1 * (b.at(v - 1) + a.v[v] + b.at(v + 1) + c.v[v]) +
                          k.c2 * (a.at(v - 1) + c.at(v - 1) + a.at(v + 1) + c.at(v + 1)) + k.cf * f[v];
        o.v[v] = row_in && in[v] ? val : 0.f;
    }
    o.sides();
}

// r = f - (20 u - 4 (W + S + E + N) - (SW + NW + SE + NE)) / (6 h^2)
template <int V>
__device__ __forceinline__ void pj_resid(const Coef& k, const Row<V>& a, const Row<V>& b, const Row<V>& c,
                                         const float (&f)[V], Row<V>& o)
{
#pragma unroll
    for (int v = 0; v < V; v++) {
        const float au = (20.f * b.v[v] - 4.f * (b.at(v - 1) + a.v[v] + b.at(v + 1) + c.v[v]) -
                          (a.at(v - 1) + c.at(v - 1) + a.at(v + 1) + c.at(v + 1))) * k.inv6h2;
        o.v[v] = f[v] - au;
    }
    o.sides();
}

// What the marching passes share: the wave's columns and rows.  Rows 0 and N-1
// and everything outside the grid count as 0 and are never read.
template <int V>
struct March {
    int N, P, x, yb, ye;               // lane's first column; rows [yb, ye) are completed
    unsigned voff;                     // its byte offset in a row, or out of range
    bool in[V], mine;                  // columns of the interior; the lane completes its columns
    __device__ __forceinline__ bool setup(int N_, int P_, int ntx, int H)
    {
        N = N_;
        P = P_;
        const unsigned tb = kg_tile_order<KG_ORD_PJ>(blockIdx.x, gridDim.x, (unsigned)ntx);
        const int lane = (int)(threadIdx.x & 63);
        const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        x = ((int)(tb % (unsigned)ntx) * MW + w) * piece<V>() + V * (lane - edge_lanes<V>());
        yb = (int)(tb / (unsigned)ntx) * H;
        ye = min(yb + H, N - 1);
        voff = x >= 0 && x < P ? (unsigned)x * 4u : kgp::KG_OOB;
#pragma unroll
        for (int v = 0; v < V; v++) in[v] = x + v >= 1 && x + v < N - 1;
        mine = lane >= edge_lanes<V>() && lane < edge_lanes<V>() + piece<V>() / V && x < P;
        return x - V * (lane - edge_lanes<V>()) < N;   // the piece has a column
    }
    __device__ __forceinline__ bool inside(int y) const { return y >= 1 && y < N - 1; }
    __device__ __forceinline__ __amdgpu_buffer_rsrc_t row(const float* p, int y) const
    {
        const bool ok = inside(y);
        return kgp::make_rsrc(p + (long long)(ok ? y : 0) * P, ok ? (unsigned)P * 4u : 0u);
    }
    __device__ __forceinline__ void load(const float* p, int y, float (&v)[V]) const
    {
        kgp::bload<kgp::F32, V>(row(p, y), voff, v);
    }
    // whole rows: interior values, 0 on the boundary and the padding
    __device__ __forceinline__ void store(float* p, int y, const Row<V>& r) const
    {
        if (mine && y >= max(yb, 1) && y < ye) {
            typedef float fv __attribute__((ext_vector_type(V)));
            fv o;
#pragma unroll
            for (int v = 0; v < V; v++) o[v] = r.v[v];
            __builtin_nontemporal_store(o, (__attribute__((address_space(1))) fv*)(p + (long long)y * P + x));
        }
    }
};

// Down: u' = two sweeps of u (ZERO: of the guess 0, which is not read) for the
// right-hand side f, and the coarse right-hand side
//   fc(I,J) = (4 r_C + 2 (r_W + r_E + r_S + r_N) + (r_SW + r_SE + r_NW + r_NE)) / 16
// of the residual r of u' at the 3 x 3 fine points around (2I, 2J).  H: even.
template <bool ZERO, int V>
__global__ __launch_bounds__(64 * MW)
void pj_down_k(int N, int P, int Nc, int Pc, int ntx, int H, Coef k, const float* __restrict__ u,
               const float* __restrict__ f, float* __restrict__ uo, float* __restrict__ fc)
{
    constexpr int D = 3;               // rows in flight
    constexpr int LAG = ZERO ? 0 : 1;  // f enters one row after u
    March<V> m;
    if (!m.setup(N, P, ntx, H)) return;
    float pu[D][V], pf[D][V], fr[3][V];
    Row<V> ur[3], s1[3], s2[3], rr[3];
#pragma unroll
    for (int q = 0; q < 3; q++) {
        ur[q] = s1[q] = s2[q] = rr[q] = Row<V>{};
#pragma unroll
        for (int v = 0; v < V; v++) fr[q][v] = 0.f;
    }
    const int first = m.yb - 3 - LAG, last = m.ye + 1 + LAG;   // incoming rows
#pragma unroll
    for (int d = 0; d < D; d++) {
        if constexpr (!ZERO) m.load(u, first + d, pu[d]);
        m.load(f, first + d - LAG, pf[d]);
    }
    // At phase p row y enters slot p; slot p+2 (mod 3) holds the row before it.
    // The first sweep's newest row is y - LAG, the second's y-1-LAG, the
    // residual's y-2-LAG; each is kept in the slot of its phase.
    auto step = [&](auto phase, int y) {
        constexpr int p = decltype(phase)::value, p1 = (p + 2) % 3, p2 = (p + 1) % 3;
#pragma unroll
        for (int v = 0; v < V; v++) fr[p][v] = pf[p][v];      // f row y - LAG
        if constexpr (ZERO) {
#pragma unroll
            for (int v = 0; v < V; v++) {
                const float val = 0.f + k.cf * fr[p][v];
                s1[p].v[v] = m.inside(y) && m.in[v] ? val : 0.f;
            }
            s1[p].sides();
        } else {
#pragma unroll
            for (int v = 0; v < V; v++) ur[p].v[v] = pu[p][v];
            ur[p].sides();
            m.load(u, y + D, pu[p]);
            pj_sweep(k, ur[p2], ur[p1], ur[p], fr[p], m.inside(y - 1), m.in, s1[p]);
        }
        m.load(f, y + D - LAG, pf[p]);
        pj_sweep(k, s1[p2], s1[p1], s1[p], fr[p1], m.inside(y - 1 - LAG), m.in, s2[p]);
        m.store(uo, y - 1 - LAG, s2[p]);
        pj_resid(k, s2[p2], s2[p1], s2[p], fr[p2], rr[p]);
        const int yr = y - 2 - LAG, J = (yr - 1) >> 1;        // residual row; its coarse row below
        if ((yr & 1) && 2 * J >= m.yb && 2 * J < m.ye && J >= 1 && J < Nc - 1) {
            const Row<V> &a = rr[p2], &b = rr[p1], &c = rr[p];
            typedef float fc_t __attribute__((ext_vector_type(V / 2)));
            float o[V / 2];
#pragma unroll
            for (int q = 0; q < V / 2; q++) {
                const int v = 2 * q, I = (m.x >> 1) + q;
                const float val = (4.f * b.v[v] + 2.f * (b.at(v - 1) + b.at(v + 1) + a.v[v] + c.v[v]) +
                                   (a.at(v - 1) + a.at(v + 1) + c.at(v - 1) + c.at(v + 1))) * 0.0625f;
                o[q] = I >= 1 && I < Nc - 1 ? val : 0.f;
            }
            if (m.mine)
                *(__attribute__((address_space(1))) fc_t*)(fc + (long long)J * Pc + (m.x >> 1)) = __builtin_bit_cast(fc_t, o);
        }
    };
    for (int y = first; y <= last; y += 3)
        kg_static_for<3>([&](auto p) {
            if (y + decltype(p)::value <= last) step(p, y + decltype(p)::value);
        });
}

// Up: u' = two sweeps of u plus the bilinear interpolation of the coarse e (e at
// even/even points, the mean of the 2 or 4 coarse neighbours elsewhere).  ADD: u'
// is not stored but added to the interior of the dense FP64 N x N field u64.
template <bool ADD, int V>
__global__ __launch_bounds__(64 * MW)
void pj_up_k(int N, int P, int Nc, int Pc, int ntx, int H, Coef k, const float* __restrict__ u,
             const float* __restrict__ ec, const float* __restrict__ f, float* __restrict__ uo,
             double* __restrict__ u64)
{
    constexpr int D = 3;
    March<V> m;
    if (!m.setup(N, P, ntx, H)) return;
    const unsigned coff = m.x >= 0 && m.x < P ? (unsigned)m.x * 2u : kgp::KG_OOB;   // column x/2
    auto crow = [&](int J, float (&v)[V / 2]) {
        const bool ok = J >= 1 && J < Nc - 1;
        kgp::bload<kgp::F32, V / 2>(kgp::make_rsrc(ec + (long long)(ok ? J : 0) * Pc, ok ? (unsigned)Pc * 4u : 0u),
                                coff, v);
    };
    float pu[D][V], pf[D][V], pa[D][V / 2], pb[D][V / 2], fr[3][V];
    Row<V> vr[3], s1[3];
#pragma unroll
    for (int q = 0; q < 3; q++) {
        vr[q] = s1[q] = Row<V>{};
#pragma unroll
        for (int v = 0; v < V; v++) fr[q][v] = 0.f;
    }
    const int first = m.yb - 2, last = m.ye + 1;
    auto fetch = [&](int y, int d) {
        m.load(u, y, pu[d]);
        m.load(f, y - 1, pf[d]);
        crow(y >> 1, pa[d]);
        crow((y >> 1) + 1, pb[d]);
    };
#pragma unroll
    for (int d = 0; d < D; d++) fetch(first + d, d);
    // N is 4 q + 1: a lane's columns, left of column N-1, are in the row
    const bool adds = m.mine && m.x < N - 1;
    d2 w[V / 2];
    auto fetch64 = [&](int y) {
        if (adds && y >= max(m.yb, 1) && y < m.ye) {
#pragma unroll
            for (int q = 0; q < V / 2; q++) w[q] = *(const d2u*)(u64 + (long long)y * N + m.x + 2 * q);
        }
    };
    auto step = [&](auto phase, int y) {
        constexpr int p = decltype(phase)::value, p1 = (p + 2) % 3, p2 = (p + 1) % 3;
        // coarse columns x/2, x/2+1 (, x/2+2) of rows y/2 and (odd y) y/2+1
        float a[V / 2 + 1], b[V / 2 + 1];
#pragma unroll
        for (int q = 0; q < V / 2; q++) {
            a[q] = pa[p][q];
            b[q] = pb[p][q];
        }
        a[V / 2] = kgp::dpp_shift<kgp::KG_DPP_WAVE_SHL1>(0.f, a[0]);
        b[V / 2] = kgp::dpp_shift<kgp::KG_DPP_WAVE_SHL1>(0.f, b[0]);
        const bool odd = y & 1;
#pragma unroll
        for (int v = 0; v < V; v++) {
            const int q = v >> 1;
            const float e = !(v & 1) ? (odd ? 0.5f * (a[q] + b[q]) : a[q])
                                     : (odd ? 0.25f * (a[q] + a[q + 1] + b[q] + b[q + 1])
                                            : 0.5f * (a[q] + a[q + 1]));
            vr[p].v[v] = m.inside(y) && m.in[v] ? pu[p][v] + e : 0.f;
            fr[p][v] = pf[p][v];                               // f row y-1
        }
        vr[p].sides();
        if constexpr (ADD) fetch64(y - 2);
        fetch(y + D, p);
        pj_sweep(k, vr[p2], vr[p1], vr[p], fr[p], m.inside(y - 1), m.in, s1[p]);
        Row<V> o;
        pj_sweep(k, s1[p2], s1[p1], s1[p], fr[p1], m.inside(y - 2), m.in, o);
        if constexpr (!ADD) {
            m.store(uo, y - 2, o);
        } else if (adds && y - 2 >= max(m.yb, 1) && y - 2 < m.ye) {
            double* q = u64 + (long long)(y - 2) * N + m.x;
#pragma unroll
            for (int h = 0; h < V / 2; h++) {
                const d2 sum = w[h] + d2{(double)o.v[2 * h], (double)o.v[2 * h + 1]};
                if (h == 0 && m.x == 0) q[1] = sum.y;          // column 0 is the caller's
                else *(d2u*)(q + 2 * h) = sum;
            }
        }
    };
    for (int y = first; y <= last; y += 3)
        kg_static_for<3>([&](auto p) {
            if (y + decltype(p)::value <= last) step(p, y + decltype(p)::value);
        });
}

// ------------------------------------------------------------ the coarse levels
// One workgroup runs the whole V-cycle from TOP cells per side (at most 128) down
// to the 2-cell level (one unknown, solved exactly) and back up, with every
// level's u in LDS and its right-hand side in the registers of the threads that
// own the points.  A thread owns R = TOP^2/1024 rows of one column (one point on
// the levels below 64 cells), so a wave reads consecutive LDS words.  As
// launches these levels took 30 of the 40 of a 512 cell V-cycle, which bound its
// solve (1.98 ms; 0.77 now).  The cycle from 128 cells takes 22 us, bound by one CU's
// FP32 rate and LDS on the first level and by barriers below.
constexpr int CTOP = 128;
constexpr int CT = 1024;               // threads
constexpr int CLV = 7;                 // levels of 128, 64, ..., 2 cells

struct CCoef {
    float c0, c1, c2, exact;           // exact: 6 h^2 / 20 of the 2-cell level
    float cf[CLV], inv6h2[CLV];        // of the levels from TOP down
};

template <int n>
struct CLevel {
    static constexpr int N = n + 1, R = n * n > CT ? n * n / CT : 1;
    static constexpr bool ONE = n <= 8;   // all points belong to the first wave, which works alone
    // Thread t's column and first row.  Column n and row n are the boundary's:
    // their threads compute along, on whatever LDS holds there, and put nothing.
    static __device__ __forceinline__ int x(int t) { return 1 + t % n; }
    static __device__ __forceinline__ int y(int t) { return 1 + t / n * R; }
    static __device__ __forceinline__ bool works(int t) { return n * n >= CT || t < n * n; }
    static __device__ __forceinline__ void sync()
    {
        if constexpr (ONE) {   // a wave's LDS operations stay in order
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        } else {
            __syncthreads();
        }
    }
    // v[r] = the thread's value of its row r / those values into a
    template <class Val>
    static __device__ __forceinline__ void each(int t, float (&v)[R], Val&& val)
    {
        const int q0 = y(t) * N + x(t);
        if (!works(t)) return;
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = val(r, q0 + r * N);
    }
    static __device__ __forceinline__ void put(int t, const float (&v)[R], float* a)
    {
        const int q0 = y(t) * N + x(t);
        if (!works(t) || x(t) == n) return;
#pragma unroll
        for (int r = 0; r < R - 1; r++) a[q0 + r * N] = v[r];
        if (y(t) + R - 1 < n) a[q0 + (R - 1) * N] = v[R - 1];
    }
    static __device__ __forceinline__ float point(const CCoef& k, float cf, const float* u, int q, float f)
    {
        return k.c0 * u[q] + k.c1 * (u[q - 1] + u[q - N] + u[q + 1] + u[q + N]) +
               k.c2 * (u[q - N - 1] + u[q + N - 1] + u[q - N + 1] + u[q + N + 1]) + cf * f;
    }
    // Two sweeps of the level in place; with zero from u = 0.
    static __device__ __forceinline__ void smooth(const CCoef& k, float cf, float* u, const float (&f)[R],
                                                  bool zero)
    {
        const int t = (int)threadIdx.x;
        float o[R] = {};
        if (zero) {
            each(t, o, [&](int r, int) { return 0.f + cf * f[r]; });
        } else {
            each(t, o, [&](int r, int q) { return point(k, cf, u, q, f[r]); });
            sync();
        }
        put(t, o, u);
        sync();
        each(t, o, [&](int r, int q) { return point(k, cf, u, q, f[r]); });
        sync();
        put(t, o, u);
        sync();
    }
    // The boundary of the level's u.
    static __device__ __forceinline__ void border(float* u)
    {
        for (int i = (int)threadIdx.x; i < N; i += CT) u[i] = u[n * N + i] = u[i * N] = u[i * N + n] = 0.f;
    }
    // One V-cycle on u (bordered; zero: u counts as 0 inside).  The memory past u
    // is the coarser levels'; d is the level's place in k.
    static __device__ __forceinline__ void cycle(const CCoef& k, int d, float* u, const float (&f)[R],
                                                 bool zero)
    {
        const int t = (int)threadIdx.x;
        if constexpr (n == 2) {
            if (t == 0) u[N + 1] = k.exact * f[0];
            sync();
        } else {
            using C = CLevel<n / 2>;
            smooth(k, k.cf[d], u, f, zero);
            float* uc = u + N * N;
            const float inv = k.inv6h2[d];
            // the residual, in the coarser levels' memory, then its restriction
            float o[R] = {};
            each(t, o, [&](int r, int q) {
                const float au = (20.f * u[q] - 4.f * (u[q - 1] + u[q - N] + u[q + 1] + u[q + N]) -
                                  (u[q - N - 1] + u[q + N - 1] + u[q - N + 1] + u[q + N + 1])) * inv;
                return f[r] - au;
            });
            put(t, o, uc);
            sync();
            float fc[C::R] = {};
            C::each(t, fc, [&](int r, int) {
                const float* p = uc + 2 * (C::y(t) + r) * N + 2 * C::x(t);
                return (4.f * p[0] + 2.f * (p[-1] + p[1] + p[-N] + p[N]) +
                        (p[-N - 1] + p[-N + 1] + p[N - 1] + p[N + 1])) * 0.0625f;
            });
            sync();
            C::border(uc);
            if constexpr (C::ONE && !ONE) {   // the border and fc of an 8-cell level are the first wave's
                if (t < 64) C::cycle(k, d + 1, uc, fc, true);
                sync();
            } else {
                C::cycle(k, d + 1, uc, fc, true);
            }
            const int xo = x(t) & 1;
            const float* e0 = uc + (x(t) >> 1);
            each(t, o, [&](int r, int q) {
                const int yy = y(t) + r;
                const float *a = e0 + (yy >> 1) * C::N, *b = a + C::N;
                const float even = xo ? 0.5f * (a[0] + a[1]) : a[0];
                const float odd = xo ? 0.25f * (a[0] + a[1] + b[0] + b[1]) : 0.5f * (a[0] + b[0]);
                return u[q] + (yy & 1 ? odd : even);
            });
            put(t, o, u);
            sync();
            smooth(k, k.cf[d], u, f, false);
        }
    }
};

template <int TOP>
__global__ __launch_bounds__(CT)
void pj_coarse_k(int P, CCoef k, const float* __restrict__ f, float* __restrict__ ug, int zero)
{
    using L = CLevel<TOP>;
    // u of the level and behind it the coarser ones, or the residual of this one,
    // and what the threads of the far boundary read past it
    __shared__ float u[2 * L::N * L::N + 2 * L::N];
    const int t = (int)threadIdx.x;
    const int o0 = L::y(t) * P + L::x(t);
    float fv[L::R] = {}, v[L::R] = {};
    L::each(t, fv, [&](int r, int) { return f[o0 + r * P]; });
    if (!zero) {
        L::each(t, v, [&](int r, int) { return ug[o0 + r * P]; });
        L::put(t, v, u);
    }
    L::border(u);
    __syncthreads();
    if (!L::ONE || t < 64) L::cycle(k, 0, u, fv, zero);
    __syncthreads();
    // interior rows, with 0 in columns 0 and N-1 (the other columns are not read)
    for (int y = 1 + (t >> 6); y < TOP; y += CT / 64)
        for (int x = t & 63; x < L::N; x += 64) ug[y * P + x] = u[y * L::N + x];
}

// The outer correction's FP64 residual, fused with its FP32 copy and its
// squared norm: r = f - (20 u - 4 (u_W + u_S + u_E + u_N) - (u_SW + u_NW +
// u_SE + u_NE)) / (6 h^2), summed in that order in FP64, written as
// FP32 rows of pitch P, 0 on the boundary columns; the sum of r^2 over the
// workgroup's points goes to part[its tile] (rows of a lane in order, then lanes
// and waves by a fixed tree).  A wave marches RES_H(n) rows of 128 columns, 2 per
// lane (rows of u start at any multiple of 8 bytes); the columns beside a lane's 2
// come by DPP, and the outer lanes only hold such columns.  Bound by HBM: 1.34 GB at
// 8192^2 in 262 us (5.1 TB/s; tiles of 8 rows with side loads from L1 289 us; 16 or
// 32 rows a wave 278 and 312).
constexpr int RPIECE = 112;   // columns a wave completes
constexpr int res_rows(int n) { return n >= 2048 ? 8 : n >= 1024 ? 4 : 2; }
constexpr int res_ntx(int n) { return (n + 1 + MW * RPIECE - 1) / (MW * RPIECE); }
constexpr int res_blocks_of(int n)
{
    return res_ntx(n) * ((n + res_rows(n) - 1) / res_rows(n));
}

__global__ __launch_bounds__(64 * MW)
void pj_residual64_k(int N, int P, int ntx, int H, double inv6h2, const double* __restrict__ u,
                     const double* __restrict__ f, float* __restrict__ r, double* __restrict__ part)
{
    constexpr int D = 3;                                       // rows in flight
    __shared__ double wsum[MW];
    const int lane = (int)(threadIdx.x & 63);
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const unsigned tb = kg_tile_order<KG_ORD_PJR>(blockIdx.x, gridDim.x, (unsigned)ntx);
    const int x = ((int)(tb % (unsigned)ntx) * MW + w) * RPIECE - 2 + 2 * lane;
    const int yb = max((int)(tb / (unsigned)ntx) * H, 1);
    const int ye = min((int)(tb / (unsigned)ntx + 1) * H, N - 1);
    // 16 bytes inside the row; what lies past an end only feeds points that are
    // not computed, except that column N-1 (even) is the second of its pair
    const int xl = min(max(x, 0), N - 2);
    const bool tail = x == N - 1;
    const bool in0 = x >= 1 && x < N - 1, in1 = x + 1 >= 1 && x + 1 < N - 1;
    const bool mine = lane >= 1 && lane <= RPIECE / 2;
    struct Row2 { double l, a, b, r; };
    Row2 ur[3];
    d2 pu[D], pf[D];
    auto row = [&](const double* p, int y) {
        return *(const d2u*)(p + (long long)min(max(y, 0), N - 1) * N + xl);
    };
    const int first = yb - 1, last = ye;                       // incoming rows of u
#pragma unroll
    for (int d = 0; d < D; d++) {
        pu[d] = row(u, first + d);
        pf[d] = row(f, first + d - 1);
        ur[d] = Row2{0.0, 0.0, 0.0, 0.0};
    }
    double acc = 0.0;
    auto step = [&](auto phase, int y) {
        constexpr int p = decltype(phase)::value, p1 = (p + 2) % 3, p2 = (p + 1) % 3;
        const d2 v = pu[p], fv = pf[p];
        pu[p] = row(u, y + D);
        pf[p] = row(f, y + D - 1);
        Row2& c = ur[p];
        c.a = tail ? v.y : v.x;
        c.b = v.y;
        c.l = kgp::dpp_shift<kgp::KG_DPP_WAVE_SHR1>(0.0, c.b);
        c.r = kgp::dpp_shift<kgp::KG_DPP_WAVE_SHL1>(0.0, c.a);
        if (y - 1 < yb) return;                                // row y-1 is the result's
        const Row2 &a = ur[p2], &b = ur[p1];
        const double au0 = (20.0 * b.a - 4.0 * (b.l + a.a + b.b + c.a) - (a.l + c.l + a.b + c.b)) * inv6h2;
        const double au1 = (20.0 * b.b - 4.0 * (b.a + a.b + b.r + c.b) - (a.a + c.a + a.r + c.r)) * inv6h2;
        const double r0 = in0 ? fv.x - au0 : 0.0, r1 = in1 ? fv.y - au1 : 0.0;
        if (mine) {
            acc += r0 * r0;
            acc += r1 * r1;
            const f2 o = {(float)r0, (float)r1};
            if (x < P) __builtin_nontemporal_store(o, (__attribute__((address_space(1))) f2*)(r + (long long)(y - 1) * P + x));
        }
    };
    for (int y = first; y <= last; y += 3)
        kg_static_for<3>([&](auto p) {
            if (y + decltype(p)::value <= last) step(p, y + decltype(p)::value);
        });
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) acc += __shfl_xor(acc, m);
    if (lane == 0) wsum[w] = acc;
    __syncthreads();
    if (threadIdx.x == 0) part[tb] = ((wsum[0] + wsum[1]) + wsum[2]) + wsum[3];
}

// out[0] = sum of part[0 .. n) in a fixed order (one workgroup of 1024
// threads: strided per-thread sums, then a tree).
__global__ __launch_bounds__(1024)
void pj_sum_k(int n, const double* __restrict__ part, double* __restrict__ out)
{
    __shared__ double t[1024];
    double s = 0.0;
    for (int i = (int)threadIdx.x; i < n; i += 8 * 1024) {   // 8 loads in flight
        double v[8];
#pragma unroll
        for (int q = 0; q < 8; q++) v[q] = i + q * 1024 < n ? part[i + q * 1024] : 0.0;
#pragma unroll
        for (int q = 0; q < 8; q++) s += v[q];
    }
    t[threadIdx.x] = s;
    __syncthreads();
    for (int m = 512; m >= 1; m >>= 1) {
        if ((int)threadIdx.x < m) t[threadIdx.x] += t[threadIdx.x + m];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = t[0];
}

// dense N x N FP64 u += FP32 rows of pitch P on the interior (a grid whose whole
// V-cycle is the coarse kernel's)
__global__ __launch_bounds__(256)
void pj_add_k(int N, int P, const float* __restrict__ e, double* __restrict__ u)
{
    const int q = (int)(blockIdx.x * 256 + threadIdx.x), j = q / N, i = q - j * N;
    if (i >= 1 && i < N - 1 && j >= 1 && j < N - 1) u[q] += (double)e[j * P + i];
}

struct Level {
    int N, P;   // vertices per side, row pitch (N rounded up to 16)
    double h;
    float *u, *t, *f;
};

// Rows per wave of the marching passes (even): the most that leaves 8 waves per
// CU, at least 2.  A wave also marches the 4 to 7 rows around its own, but on
// small levels its latency is what counts: a 512 cell solve takes 1.20 ms at 8 rows,
// 1.07 at 4, 1.03 at 2; at 8192 cells 16 to 24 rows are the best of 8 .. 128 by 2 %.
int march_rows(const kg_ctx* ctx, int ntx, int N)
{
    for (int H : {16, 8, 4})
        if ((long long)ntx * ((N - 2) / H + 1) >= 2LL * ctx->cus) return H;
    return 2;
}

constexpr double OMEGA = 0.8;   // damping; two sweeps before and two after the coarse levels

float sweep_cf(double h) { return (float)(3 * OMEGA * h * h / 10); }
float residual_scale(double h) { return (float)(1.0 / (6.0 * h * h)); }
constexpr float C0 = (float)(1 - OMEGA), C1 = (float)(OMEGA / 5), C2 = (float)(OMEGA / 20);

template <int TOP>
void launch_coarse(hipStream_t st, const Level& L, bool zero)
{
    CCoef k{};
    k.c0 = C0;
    k.c1 = C1;
    k.c2 = C2;
    k.exact = (float)(6.0 * 0.5 * 0.5 / 20.0);
    int d = 0;
    for (int n = TOP; n > 2; n /= 2, d++) {
        k.cf[d] = sweep_cf(1.0 / n);
        k.inv6h2[d] = residual_scale(1.0 / n);
    }
    hipLaunchKernelGGL(pj_coarse_k<TOP>, dim3(1), dim3(CT), 0, st, L.P, k, (const float*)L.f, L.u,
                       (int)zero);
}

// One V-cycle on level l from its u (zero: from 0), which ends in L.u, or, with
// u64, is added to that field.  Rows 0 and N-1 of the levels' arrays are never
// read or written.
void vcycle(const kg_ctx* ctx, hipStream_t st, Level* lv, int l, bool zero, double* u64)
{
    Level& L = lv[l];
    if (L.N - 1 <= CTOP) {
        switch (L.N - 1) {
        case 2: launch_coarse<2>(st, L, zero); break;
        case 4: launch_coarse<4>(st, L, zero); break;
        case 8: launch_coarse<8>(st, L, zero); break;
        case 16: launch_coarse<16>(st, L, zero); break;
        case 32: launch_coarse<32>(st, L, zero); break;
        case 64: launch_coarse<64>(st, L, zero); break;
        default: launch_coarse<CTOP>(st, L, zero); break;
        }
        if (u64)
            hipLaunchKernelGGL(pj_add_k, dim3((unsigned)((L.N * L.N + 255) / 256)), dim3(256), 0, st, L.N,
                               L.P, (const float*)L.u, u64);
        return;
    }
    Level& C = lv[l + 1];
    const Coef k{C0, C1, C2, sweep_cf(L.h), residual_scale(L.h)};
    const int ntx4 = (L.N + MW * piece<4>() - 1) / (MW * piece<4>());
    const int H = march_rows(ctx, ntx4, L.N);
    const bool narrow = H == 2;
    const int ntx = narrow ? (L.N + MW * piece<2>() - 1) / (MW * piece<2>()) : ntx4;
    const unsigned blocks = (unsigned)ntx * (unsigned)((L.N - 1 + H - 1) / H);
    auto down = narrow ? (zero ? pj_down_k<true, 2> : pj_down_k<false, 2>)
                       : (zero ? pj_down_k<true, 4> : pj_down_k<false, 4>);
    hipLaunchKernelGGL(down, dim3(blocks), dim3(64 * MW), 0, st, L.N, L.P, C.N, C.P, ntx, H, k,
                       (const float*)L.u, (const float*)L.f, L.t, C.f);
    std::swap(L.u, L.t);
    vcycle(ctx, st, lv, l + 1, true, nullptr);
    auto up = narrow ? (u64 ? pj_up_k<true, 2> : pj_up_k<false, 2>) : (u64 ? pj_up_k<true, 4> : pj_up_k<false, 4>);
    hipLaunchKernelGGL(up, dim3(blocks), dim3(64 * MW), 0, st, L.N, L.P, C.N, C.P, ntx, H, k,
                       (const float*)L.u, (const float*)C.u, (const float*)L.f, L.t, u64);
    std::swap(L.u, L.t);
}

// Levels n, n/2, ..., 2 cells per side: at most 14 for n <= 16384.
constexpr int MAX_LEVELS = 14;
constexpr int MAX_N = 1 << 14;

// Device memory of one solve, carved in a fixed order from one or more
// regions: per level (finest first) u, t and f (N x P floats each), then the
// residual pass's partial sums (res_blocks + 1 doubles), then the partials of
// the norm of f (kg_stats_scratch_bytes()).  Every block starts at a
// multiple of 256 bytes.
struct Workspace {
    int nl;
    Level lv[MAX_LEVELS];
    int res_blocks;
    double* part;
    double* stats;
};

constexpr size_t align256(size_t b) { return (b + 255) / 256 * 256; }
constexpr int pitch(int N) { return (N + 15) / 16 * 16; }
// Bytes of the workspace of an n-cell solve (n a power of two >= 2).
constexpr size_t workspace_bytes(int n, size_t stats_bytes)
{
    size_t b = 0;
    for (int m = n; m >= 2; m /= 2) {
        const size_t ne = (size_t)(m + 1) * (size_t)pitch(m + 1);
        b += 3 * align256(ne * sizeof(float));
    }
    b += align256((size_t)(res_blocks_of(n) + 1) * sizeof(double));
    b += align256(stats_bytes);
    return b;
}

// Level sizes of an n-cell solve; pointers left null.
void workspace_shape(Workspace& ws, int n)
{
    ws.nl = 0;
    for (int m = n; m >= 2; m /= 2)
        ws.lv[ws.nl++] = Level{m + 1, pitch(m + 1), 1.0 / m, nullptr, nullptr, nullptr};
    ws.res_blocks = res_blocks_of(n);
    ws.part = ws.stats = nullptr;
}

// Points the workspace's blocks into the region at base (workspace_bytes(n)
// bytes, 256-byte aligned).
void workspace_carve(Workspace& ws, char* base)
{
    size_t off = 0;
    for (int l = 0; l < ws.nl; l++) {
        Level& L = ws.lv[l];
        const size_t b = align256((size_t)L.N * L.P * sizeof(float));
        for (float** p : {&L.u, &L.t, &L.f}) {
            *p = (float*)(base + off);
            off += b;
        }
    }
    ws.part = (double*)(base + off);
    off += align256((size_t)(ws.res_blocks + 1) * sizeof(double));
    ws.stats = (double*)(base + off);
}

int check_args(kg_ctx* ctx, const char* who, int n, int nmax, const double* f, const double* u)
{
    if (int rc = kg_check_ctx(ctx)) return rc;
    if (n < 2 || (n & (n - 1)) || n > nmax)
        return kg_set_error(KG_ERR_INVALID, "%s: n = %d must be a power of two in [2, %d]", who, n, nmax);
    if (!f || !u) return kg_set_error(KG_ERR_INVALID, "%s: null buffer", who);
    if ((const void*)f == (const void*)u)
        return kg_set_error(KG_ERR_INVALID, "%s: f and u must be distinct", who);
    return KG_OK;
}

// The defect-correction loop on a carved workspace (of any contents); the stream
// is synchronised on return.  Timing (events or the host clock) is the
// caller's: t_start is called once the norm of f is known, right before the
// first residual pass.
template <class Start>
int solve(kg_ctx* ctx, int n, const double* f, double* u, double tol, int max_outer, int vcycles,
          Workspace& ws, kg_poisson_report* rep, int* outer_out, int* cycles_out, double* rel_out,
          Start&& t_start)
{
    hipStream_t st = kg_stream(ctx);
    const int N = n + 1;
    const long long np = (long long)N * N;
    const double h = 1.0 / n;
    if (max_outer < 1) max_outer = 1;
    if (vcycles < 1) vcycles = 1;
    double st_f[5];
    const bool host = ctx->host != nullptr;   // where the results come to
    double* stats = host ? ctx->host : ws.stats + kg_stats_scratch_bytes() / sizeof(double) - 5;
    double* sum = host ? ctx->host : ws.part + ws.res_blocks;
    if (int rc = kg_field_stats_launch(st, KG_F64, (size_t)np, f, KG_F64, nullptr, ws.stats, stats)) return rc;
    if (int rc = kg_bring_results(st, st_f, stats, 5, host)) return rc;
    const double fnorm = std::sqrt(st_f[1]);
    int outer = 0, cycles = 0;
    double rel = 0;
    Level& F = ws.lv[0];
    t_start();
    for (;;) {
        // r = f - A u in FP64: its FP32 copy is the right-hand side of the
        // inner solve (F.f), its squared norm decides the stop
        hipLaunchKernelGGL(pj_residual64_k, dim3(ws.res_blocks), dim3(64 * MW), 0, st, N, F.P,
                           res_ntx(n), res_rows(n), 1.0 / (6.0 * h * h), (const double*)u, f, F.f, ws.part);
        hipLaunchKernelGGL(pj_sum_k, dim3(1), dim3(1024), 0, st, ws.res_blocks,
                           (const double*)ws.part, sum);
        double sumsq = 0.0;
        if (int rc = kg_bring_results(st, &sumsq, sum, 1, host)) return rc;
        rel = fnorm > 0 ? std::sqrt(sumsq) / fnorm : 0.0;
        if (rep && outer < KG_POISSON_HISTORY) rep->history[outer] = rel;
        if (rel < tol || outer >= max_outer) break;
        // inner FP32 solve of A e = r from e = 0, then u += e
        for (int c = 0; c < vcycles; c++)
            vcycle(ctx, st, ws.lv, 0, c == 0, c == vcycles - 1 ? u : nullptr);
        cycles += vcycles;
        outer++;
    }
    KG_HIP(hipGetLastError());
    *outer_out = outer;
    *cycles_out = cycles;
    *rel_out = rel;
    return KG_OK;
}

int finish(const char* who, kg_poisson_report* rep, const Workspace& ws, int outer, int cycles,
           double rel, double seconds, double tol)
{
    if (rep) {
        rep->outer = outer;
        rep->vcycles = cycles;
        rep->rel_residual = rel;
        rep->seconds = seconds;
        rep->levels = ws.nl;
    }
    return rel < tol ? KG_OK : kg_set_error(KG_ERR_STATE, "%s: relative residual %.3e after %d "
                                            "corrections (tol %.1e)", who, rel, outer, tol);
}

// ---- the static workspace of kg_poisson_solve_noalloc ----------------------
// Sized for the largest grid that entry point accepts; one copy per device
// (a __device__ array exists once on every GPU the code object is loaded
// on), held until the process ends.
constexpr int NOALLOC_MAX_N = KG_POISSON_NOALLOC_MAX_N;
constexpr size_t STATS_BYTES = (1024 * 5 + 5) * sizeof(double);   // kg_stats_scratch_bytes()
constexpr size_t NOALLOC_BYTES = workspace_bytes(NOALLOC_MAX_N, STATS_BYTES);

constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
char* g_scratch_ptr[MAX_DEVICES];   // device address of `scratch` on each device, once set up

}  // namespace

static __device__ __align__(256) unsigned char scratch[NOALLOC_BYTES];

// Called by kg_init with `device` current: looks up this device's copy of
// the static workspace once.  Host code uses only the address found here;
// `scratch` itself names a host-side stand-in.
int kg_poisson_static_setup(int device)
{
    if (device < 0 || device >= MAX_DEVICES)
        return kg_set_error(KG_ERR_NODEV, "kg_poisson_static_setup: device %d beyond %d", device, MAX_DEVICES);
    if (kg_stats_scratch_bytes() != STATS_BYTES)
        return kg_set_error(KG_ERR_STATE, "kg_poisson_static_setup: statistics scratch size mismatch");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[device]) return KG_OK;
    void* p = nullptr;
    KG_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p || ((uintptr_t)p & 255))
        return kg_set_error(KG_ERR_HIP, "kg_poisson_static_setup: bad workspace address %p", p);
    g_scratch_ptr[device] = (char*)p;
    return KG_OK;
}

extern "C" int kg_poisson_solve(kg_ctx* ctx, int n, const double* f, double* u, double tol,
                                int max_outer, int vcycles, kg_poisson_report* rep)
{
    if (int rc = check_args(ctx, "kg_poisson_solve", n, MAX_N, f, u)) return rc;
    KG_HIP(hipSetDevice(ctx->device));
    hipStream_t st = kg_stream(ctx);
    Workspace ws;
    workspace_shape(ws, n);
    const size_t bytes = workspace_bytes(n, kg_stats_scratch_bytes());
    char* base = nullptr;
    hipError_t e = hipMalloc((void**)&base, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return kg_set_error(KG_ERR_NOMEM, "kg_poisson_solve: %zu bytes: %s", bytes, hipGetErrorString(e));
    }
    hipEvent_t e0 = nullptr, e1 = nullptr;
    // every exit from here on waits for the stream and releases what was taken
    auto done = [&](int rc) {
        (void)hipStreamSynchronize(st);
        if (e0) (void)hipEventDestroy(e0);
        if (e1) (void)hipEventDestroy(e1);
        (void)hipFree(base);
        return rc;
    };
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
        (void)hipGetLastError();
        return done(kg_set_error(KG_ERR_HIP, "kg_poisson_solve: hipEventCreate failed"));
    }
    workspace_carve(ws, base);
    kg_register_kernel("poisson_smooth", (const void*)pj_up_k<false, 4>);
    int outer = 0, cycles = 0;
    double rel = 0;
    if (int rc = solve(ctx, n, f, u, tol, max_outer, vcycles, ws, rep, &outer, &cycles, &rel,
                       [&] { (void)hipEventRecord(e0, st); }))
        return done(rc);
    float ms = 0;
    if (hipEventRecord(e1, st) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
        hipEventElapsedTime(&ms, e0, e1) != hipSuccess) {
        (void)hipGetLastError();
        return done(kg_set_error(KG_ERR_HIP, "kg_poisson_solve: event timing failed"));
    }
    return done(finish("kg_poisson_solve", rep, ws, outer, cycles, rel, ms * 1e-3, tol));
}

extern "C" int kg_poisson_solve_noalloc(kg_ctx* ctx, int n, const double* f, double* u, double tol,
                                        int max_outer, int vcycles, kg_poisson_report* rep)
{
    if (int rc = check_args(ctx, "kg_poisson_solve_noalloc", n, NOALLOC_MAX_N, f, u)) return rc;
    if (ctx->device < 0 || ctx->device >= MAX_DEVICES || !g_scratch_ptr[ctx->device])
        return kg_set_error(KG_ERR_STATE, "kg_poisson_solve_noalloc: workspace of device %d not set up",
                            ctx->device);
    KG_HIP(hipSetDevice(ctx->device));
    hipStream_t st = kg_stream(ctx);
    Workspace ws;
    workspace_shape(ws, n);
    if (workspace_bytes(n, STATS_BYTES) > NOALLOC_BYTES)
        return kg_set_error(KG_ERR_INVALID, "kg_poisson_solve_noalloc: n = %d needs %zu bytes of "
                            "workspace, more than the %zu reserved", n, workspace_bytes(n, STATS_BYTES),
                            NOALLOC_BYTES);
    workspace_carve(ws, g_scratch_ptr[ctx->device]);
    kg_register_kernel("poisson_smooth", (const void*)pj_up_k<false, 4>);
    int outer = 0, cycles = 0;
    double rel = 0;
    std::chrono::steady_clock::time_point t0;
    int rc = solve(ctx, n, f, u, tol, max_outer, vcycles, ws, rep, &outer, &cycles, &rel,
                   [&] { t0 = std::chrono::steady_clock::now(); });
    (void)hipStreamSynchronize(st);
    if (rc) return rc;
    const double sec = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    return finish("kg_poisson_solve_noalloc", rep, ws, outer, cycles, rel, sec, tol);
}

int kg_preload_poisson() { return kg_preload_kernel((const void*)pj_up_k<false, 4>); }
