// kg_matmul.hip -- C(nx,ns) += A(nx,ny) * B(ny,ns), column-major FP64, on
// the FP64 matrix cores (v_mfma_f64_16x16x4f64).  The suite's only dense
// contraction (matmul/matmul.F90:56-68).
//
// At the benchmark shape (512 x 256 x 256, 67 MFLOP) the step is latency
// work, not throughput work: at the FP64 matrix peak it is under a
// microsecond.  So the kernel for such products (matmul_k) is shaped for many
// short, independent waves whose loads are all in flight before the first product
// (larger ones: matmul_tiles_k):
//
//   * a workgroup of KS = 4 waves owns one 16 x 16 tile of C (512 workgroups
//     at 512 x 256: two per compute unit);
//   * wave w takes k in [w*kq, (w+1)*kq), kq = ny/KS rounded up to a
//     multiple of 4, in chunks of KC = 64 (16 MFMA steps); every operand of a
//     chunk is loaded into registers before its first MFMA;
//   * the MFMA step s of a chunk uses the four k values k0 + 2*(l/16) + s%2 +
//     8*(s/2) of lane group l/16 (any four distinct k form a valid step), so
//     the B operands of steps 2t and 2t+1 are one 16-byte load of the
//     contiguous pair B(k, j), B(k+1, j) (B is k-contiguous);
//   * waves 1..3 leave their partial tiles in LDS and wave 0 adds them to
//     its own in that fixed order (the result does not depend on timing),
//     then writes C.
//
// Lane l supplies A(i0 + l%16, k) and B(k, j0 + l%16); its four accumulators
// are C(i0 + l/16 + 4*r, j0 + l%16), r = 0..3 (the accumulator layout of the
// instruction, checked on the device).  Products outside the matrices are
// zero.  Sums are formed by the matrix core in blocks of four fused products
// and the four k ranges are added at the end, so the result differs from a
// strictly sequential k loop by rounding (bounded norm-wise).
#include "kg_internal.h"

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));
typedef double v2u __attribute__((ext_vector_type(2), aligned(8)));   // at any element

// Measured at 512 x 256 x 256 (40 back-to-back launches): 8.1 us (8.3
// TFLOP/s) against 61 us for one wave per tile walking all of k with each
// load waited for before its product; k split 2 ways 10.0 us, 8 ways 8.6,
// 16 ways 8.3, 64-k or 32-k chunks alike.
#ifndef KG_MM_KS
#define KG_MM_KS 4
#endif
#ifndef KG_MM_KC
#define KG_MM_KC 64
#endif
#ifndef KG_ORD_MM
#define KG_ORD_MM 8            // 2048^3: 2 or 4 2 % slower
#endif
constexpr int KS = KG_MM_KS;   // waves per workgroup: the k range split KS ways
constexpr int KC = KG_MM_KC;   // k values per chunk (KC/4 MFMA steps)
constexpr int STEPS = KC / 4;

__global__ __launch_bounds__(64 * KS)
void matmul_k(int nx, int ny, int ns, int ntile_i, int kq, const double* __restrict__ A,
              const double* __restrict__ B, double* __restrict__ C)
{
    __shared__ v4d part[KS - 1][64];
    const int wave = (int)(threadIdx.x >> 6);
    const int lane = (int)(threadIdx.x & 63);
    const int i0 = (int)(blockIdx.x % (unsigned)ntile_i) * 16;
    const int j0 = (int)(blockIdx.x / (unsigned)ntile_i) * 16;
    const int lr = lane & 15;        // row of A / column of B and C within the tile
    const int lg = lane >> 4;        // lane group 0..3
    const int ia = i0 + lr, jb = j0 + lr;
    const bool a_ok = ia < nx, b_ok = jb < ns;
    const double* Arow = A + ia;
    const double* Bcol = B + (long long)ny * jb;
    // B pairs are 16-byte loads when every column starts 16-byte aligned
    const bool b16 = !(ny & 1) && !((uintptr_t)B & 15);

    v4d acc = {0.0, 0.0, 0.0, 0.0};
    if (wave == 0) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int i = i0 + lg + 4 * r;
            acc[r] = (i < nx && b_ok) ? C[(long long)i + (long long)nx * jb] : 0.0;
        }
    }
    const int kb = wave * kq, ke = min(kb + kq, ny);
    for (int k0 = kb; k0 < ke; k0 += KC) {
        double av[STEPS], bv[STEPS];
#pragma unroll
        for (int t = 0; t < STEPS / 2; t++) {
            const int k = k0 + 8 * t + 2 * lg;   // this lane group's pair k, k+1
            const bool k0ok = k < ke, k1ok = k + 1 < ke;
            av[2 * t] = (a_ok && k0ok) ? Arow[(long long)nx * k] : 0.0;
            av[2 * t + 1] = (a_ok && k1ok) ? Arow[(long long)nx * (k + 1)] : 0.0;
            if (b16 && b_ok && k1ok) {
                const v2d p = *(const v2d*)(Bcol + k);
                bv[2 * t] = p[0];
                bv[2 * t + 1] = p[1];
            } else {
                bv[2 * t] = (b_ok && k0ok) ? Bcol[k] : 0.0;
                bv[2 * t + 1] = (b_ok && k1ok) ? Bcol[k + 1] : 0.0;
            }
        }
#pragma unroll
        for (int s = 0; s < STEPS; s++)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av[s], bv[s], acc, 0, 0, 0);
    }
    if (wave > 0) part[wave - 1][lane] = acc;
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int w = 0; w < KS - 1; w++) acc += part[w][lane];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int i = i0 + lg + 4 * r;
        if (i < nx && b_ok) C[(long long)i + (long long)nx * jb] = acc[r];
    }
}

// Tiles of 16 T x 16 T (T = 2 or 4) for products large enough to fill the device
// with them: every wave of the 4 holds the whole tile for its k range (the ranges,
// their blocks of four products and the order in which they are added are
// matmul_k's, and so is the result, bit for bit), so an operand read feeds T matrix
// steps instead of one.  An MFMA step occupies its SIMD for 64 cycles: at T = 4 the
// 16 of a k block take 1024 cycles for 4 KB of operands, which the caches deliver
// straight into registers, 8 values of k ahead (a wave's next operands have 2048
// cycles to arrive).  LDS only serves the final sum, in T T / 4 tiles at a time.
//
// Row m of tile 2p+q is row 32p + 2m + q: the operands of two tiles are one 16-byte
// load of A, and a lane's results are pairs of rows.  Rows and columns past the
// matrix read its last ones and are not stored.
//
// 2048^3 261 us (65.7 TFLOP/s), bound by the matrix cores, against 680 with 16 x 16
// tiles, whose operand reads bound it; 1500^3 153 us (429), 1024^3 43 (91); launches queued
// behind each other, 2048^3 waited for alone 280.  T = 2
// reaches 44 TFLOP/s at 2048^3, bound by L1 (2 to 4 blocks in flight change nothing),
// but gives a smaller product four times as many workgroups: 512 x 512 with k =
// 2048 30 us (72 with T = 4, 48 with 16 x 16 tiles), 512^3 9.5 (24 and 15).
template <int T>
__global__ __launch_bounds__(64 * KS, T == 2 ? 6 : 2)
void matmul_tiles_k(int nx, int ny, int ns, int ntile_i, int kq, const double* __restrict__ A,
                    const double* __restrict__ B, double* __restrict__ C)
{
    constexpr int Q = T * T / KS;      // 16 x 16 tiles a wave sums and stores
    __shared__ v4d part[KS][Q][64];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = (int)(threadIdx.x & 63);
    const int lr = lane & 15, lg = lane >> 4;
    const unsigned tb = kg_tile_order<KG_ORD_MM>(blockIdx.x, gridDim.x, (unsigned)ntile_i);
    const int i0 = (int)(tb % (unsigned)ntile_i) * 16 * T, j0 = (int)(tb / (unsigned)ntile_i) * 16 * T;
    const int kb = wave * kq, ke = min(kb + kq, ny);

    v4d acc[T][T];
#pragma unroll
    for (int a = 0; a < T; a++)
#pragma unroll
        for (int b = 0; b < T; b++) {
            const int j = j0 + 16 * b + lr;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int i = i0 + 32 * (a / 2) + 2 * (lg + 4 * r) + a % 2;
                acc[a][b][r] = wave == 0 && i < nx && j < ns ? C[(long long)i + (long long)nx * j] : 0.0;
            }
        }

    const double *pa[T / 2], *pb[T];   // operands of k = kb + 2 lg
    bool tail[T / 2];                  // the lane's first row is the matrix's last
#pragma unroll
    for (int p = 0; p < T / 2; p++) {
        const int i = i0 + 32 * p + 2 * lr;
        tail[p] = i == nx - 1;
        pa[p] = A + min(i, nx - 2) + (long long)nx * (kb + 2 * lg);
    }
#pragma unroll
    for (int b = 0; b < T; b++) pb[b] = B + (long long)ny * min(j0 + 16 * b + lr, ns - 1) + kb + 2 * lg;

    struct Ops { v2d a[T / 2][2], b[T]; };   // two MFMA steps: 8 values of k
    Ops next;
    auto load = [&](Ops& o) {
#pragma unroll
        for (int p = 0; p < T / 2; p++) {
            o.a[p][0] = *(const v2u*)pa[p];
            o.a[p][1] = *(const v2u*)(pa[p] + nx);
            pa[p] += 8LL * nx;
        }
#pragma unroll
        for (int b = 0; b < T; b++) {
            o.b[b] = *(const v2u*)pb[b];
            pb[b] += 8;
        }
    };
    auto mult = [&](const Ops& o) {
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int p = 0; p < T / 2; p++) {
                const double x = o.a[p][s].x, y = o.a[p][s].y;
                const double a0 = tail[p] ? y : x;
#pragma unroll
                for (int b = 0; b < T; b++) {
                    acc[2 * p][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, o.b[b][s], acc[2 * p][b], 0, 0, 0);
                    acc[2 * p + 1][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(y, o.b[b][s], acc[2 * p + 1][b], 0, 0, 0);
                }
            }
    };
    const int nt = ke > kb ? (ke - kb) / 8 : 0;
    if (nt > 0) load(next);
    for (int t = 0; t < nt; t++) {
        const Ops o = next;
        if (t + 1 < nt) load(next);
        mult(o);
    }
    if (kb + 8 * nt < ke) {            // the last 1 .. 7 values: 0 past them
        const int k = kb + 8 * nt + 2 * lg;
        const bool k0ok = k < ke, k1ok = k + 1 < ke;
        Ops o;
#pragma unroll
        for (int p = 0; p < T / 2; p++) {
            o.a[p][0] = o.a[p][1] = v2d{0.0, 0.0};
            if (k0ok) o.a[p][0] = *(const v2u*)pa[p];
            if (k1ok) o.a[p][1] = *(const v2u*)(pa[p] + nx);
        }
#pragma unroll
        for (int b = 0; b < T; b++) {
            o.b[b].x = k0ok ? pb[b][0] : 0.0;
            o.b[b].y = k1ok ? pb[b][1] : 0.0;
        }
        mult(o);
    }

    // the four ranges' sums, in order; wave w adds and stores tiles w Q .. w Q + Q-1
    kg_static_for<KS>([&](auto c) {
        constexpr int w = decltype(c)::value;
        if (w > 0) __syncthreads();
        if (wave != w) {
#pragma unroll
            for (int q = 0; q < Q; q++) part[wave][q][lane] = acc[(w * Q + q) / T][(w * Q + q) % T];
        }
        __syncthreads();
        if (wave == w) {
#pragma unroll
            for (int q = 0; q < Q; q++) {
                const int a = (w * Q + q) / T, b = (w * Q + q) % T;
                v4d sum = w == 0 ? acc[a][b] : part[0][q][lane];
#pragma unroll
                for (int v = 1; v < KS; v++) sum += v == w ? acc[a][b] : part[v][q][lane];
                const int j = j0 + 16 * b + lr;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int i = i0 + 32 * (a / 2) + 2 * (lg + 4 * r) + a % 2;
                    if (i < nx && j < ns) C[(long long)i + (long long)nx * j] = sum[r];
                }
            }
        }
    });
}

template <int T>
void launch_tiles(kg_ctx* ctx, int nx, int ny, int ns, int kq, const double* A, const double* B, double* C)
{
    const int ti = (nx + 16 * T - 1) / (16 * T), tj = (ns + 16 * T - 1) / (16 * T);
    kg_launch(ctx, matmul_tiles_k<T>, dim3((unsigned)((long long)ti * tj)), dim3(64 * KS), 0, nx, ny, ns, ti,
              kq, A, B, C);
}

// The work of the busiest CU in 16 x 16 tiles when it is dealt out in tiles of T x T.
long long busiest(const kg_ctx* ctx, int nx, int ns, int T)
{
    const long long t = (long long)((nx + 16 * T - 1) / (16 * T)) * ((ns + 16 * T - 1) / (16 * T));
    return (t + ctx->cus - 1) / ctx->cus * T * T;
}

// Tile edge in units of 16.  A 16 x 16 tile of the result costs its CU 2.2, 3.0 and
// 5.3 us per 1000 values of k at T = 4, 2 and 1, so a larger T is taken unless it leaves
// the busiest CU too much: T = 4 up to 4/3 of T = 2 (equal times at 777 x 1333 x 901,
// 16 against 12; at 301 x 2011 x 1203, 16 against 8, T = 2 is 1.4 times as fast),
// T = 2 below twice T = 1 (3 against 4 at 333 x 257 x 421: 7.9 against 10.5 us; 2
// against 4 at 512 x 256 x 256: 7.3 against 6.3).
int tile_edge(const kg_ctx* ctx, int nx, int ns)
{
    const long long w1 = busiest(ctx, nx, ns, 1), w2 = busiest(ctx, nx, ns, 2), w4 = busiest(ctx, nx, ns, 4);
    if (nx < 2 || w2 >= 2 * w1) return 1;   // (pairs of rows)
    return 3 * w4 <= 4 * w2 ? 4 : 2;
}

}  // namespace

extern "C" int kg_matmul(kg_ctx* ctx, int nx, int ny, int ns, const double* A, const double* B,
                         double* C)
{
    if (int rc = kg_check_ctx(ctx)) return rc;
    if (nx < 0 || ny < 0 || ns < 0)
        return kg_set_error(KG_ERR_INVALID, "kg_matmul: negative dimension (%d, %d, %d)", nx, ny, ns);
    if (!A || !B || !C) return kg_set_error(KG_ERR_INVALID, "kg_matmul: null buffer");
    if (C == A || C == B) return kg_set_error(KG_ERR_INVALID, "kg_matmul: C aliases an input");
    const int ti = (nx + 15) / 16, tj = (ns + 15) / 16;
    const long long tiles = (long long)ti * tj;
    if (tiles > 0xFFFFFFFFLL / 256)
        return kg_set_error(KG_ERR_INVALID, "kg_matmul: %lld tiles exceed one launch", tiles);
    // each wave's k range: a quarter of ny rounded up to whole MFMA steps
    const int kq = ((ny + KS - 1) / KS + 3) / 4 * 4;
    const int edge = tile_edge(ctx, nx, ns);
    kg_register_kernel("matmul_", edge == 4 ? (const void*)matmul_tiles_k<4>
                                : edge == 2 ? (const void*)matmul_tiles_k<2> : (const void*)matmul_k);
    if (int rc = kg_launch_begin(ctx, "matmul_")) return rc;
    if (edge == 4) launch_tiles<4>(ctx, nx, ny, ns, kq, A, B, C);
    else if (edge == 2) launch_tiles<2>(ctx, nx, ny, ns, kq, A, B, C);
    else if (tiles > 0)
        kg_launch(ctx, matmul_k, dim3((unsigned)tiles), dim3(64 * KS), 0, nx, ny, ns, ti, kq, A, B,
                  C);
    return kg_launch_end(ctx);
}

int kg_preload_matmul() { return kg_preload_kernel((const void*)matmul_k); }
