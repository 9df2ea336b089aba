// Format B: one uint8 code per weight, one 256-entry fp32 codebook per 64
// consecutive output rows.  y[o] = sum_k cb[o/64][W[o,k]] * x[k].
//
// The format has no reference function (its nearest analogue is the byte-LUT
// decode of crates/needle-core/src/cq.rs:838-873); the semantics are the
// closed form above.
//
// GEMV (decode, batch 1) is HBM-bound: 1 byte of code per multiply-add, so
// the kernel is shaped around keeping HBM streaming while each code costs a
// byte extract, an LDS gather and one FMA:
//   * one 64-row codebook tile per 4-wave workgroup, 32 lanes per row, the
//     lane's activations in registers (fast path: in = 256*M);
//   * the codebook in LDS as 32 lane-private replicas, so random gathers do
//     not conflict on banks;
//   * code loads split in two halves so the second half is in flight while
//     the first computes; nontemporal loads, since codes are read once.
// Other widths take a kernel with the activations in LDS and part steps.
// GEMM (prefill) rounds X to bf16, dequantises weights to bf16 through the
// bf16-rounded codebook and feeds v_mfma_f32_16x16x32_bf16 with fp32
// accumulation: up to 64 rows, and for launches too small to fill the chip,
// codes go from memory to fragments in 64x128 tiles; above, weight tiles go
// through LDS, 128x128, and 256x256 with two waves per SIMD once a launch has a
// tile per CU.
#include "nd_internal.h"
#include "nd_lanes.h"

#include <hip/hip_bf16.h>

namespace {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr int kTileRows = 64;      // rows sharing one codebook
constexpr int kThreads = 256;      // 4 waves

// Fast path, in = 256*M (M = 1..4; config 1's 768 is M = 3).  One 256-thread
// block owns one 64-row tile.  32 lanes share a row: lane j reads M/2
// 16-byte vectors (bytes 512k + 16j) and, for odd M, one 8-byte vector
// (bytes 512*(M/2) + 8j) -- every load instruction covers two rows x 256 or
// 512 contiguous bytes -- and keeps the matching 8*M activations in
// registers.  A wave's 16 rows (8 passes of two) are all loaded before the
// first gather.  Each pass leaves one partial a lane; the 8 partials are
// summed over their half waves together at the end with VALU lane moves
// (a per-pass shuffle reduction costs five LDS round trips a row, which
// measured 72-75 % of HBM against 85 % for the deferred sum).  Rows past
// `out` are clamped (a valid row is read and its sum discarded) rather than
// predicated.
//
// The codebook sits in LDS as 32 lane-private replicas, entry-major (entry
// e, replica r at dword 32e + r): lane l's gathers all hit bank l % 32, so a
// random gather does not conflict.
template <int M>
struct RowCodes {
    u32x4_t a[M / 2 > 0 ? M / 2 : 1];
    u32x2_t b;
};

template <int M>
__device__ inline void load_row(RowCodes<M> &c, const uint8_t *__restrict__ rp, int j)
{
#pragma unroll
    for (int k = 0; k < M / 2; ++k)
        c.a[k] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t *>(rp + 512 * k) + j);
    if (M % 2)
        c.b = __builtin_nontemporal_load(reinterpret_cast<const u32x2_t *>(rp + 512 * (M / 2)) + j);
}

template <int M>
__global__ __launch_bounds__(kThreads, 4) void cb8_gemv_kernel(
    const uint8_t *__restrict__ w, size_t w_stride, const float *__restrict__ cb,
    size_t cb_stride, const float *__restrict__ x, size_t x_stride, float *__restrict__ y,
    size_t y_stride, int out)
{
    constexpr int K = 256 * M;
    constexpr int kPasses = 8;  // 16 rows per wave, 2 per pass
    constexpr int kFirst = kPasses;
    __shared__ float4 rep4[256 * 32 / 4];  // 32 KB

    const size_t prob = blockIdx.y;
    w += prob * w_stride;
    cb += prob * cb_stride + size_t(blockIdx.x) * 256;
    x += prob * x_stride;
    y += prob * y_stride;
    const int t = threadIdx.x;
    const int wave = t >> 6;
    const int lane = t & 63;
    const int j = lane & 31;
    const int row0 = blockIdx.x * kTileRows + wave * 16 + (lane >> 5);

    RowCodes<M> c[kPasses];
#pragma unroll
    for (int p = 0; p < kFirst; ++p) {
        const int r = min(row0 + 2 * p, out - 1);
        load_row(c[p], w + size_t(r) * K, j);
    }
    // float4 slot f4 = i*256 + t of the replica array holds entry f4 / 8.
    float cbv[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) cbv[i] = cb[(i * kThreads + t) >> 3];
    float xa[M / 2 > 0 ? M / 2 : 1][16], xb[8];
#pragma unroll
    for (int k = 0; k < M / 2; ++k) {
        const float4 *xp = reinterpret_cast<const float4 *>(x + 512 * k + 16 * j);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 v = xp[q];
            xa[k][4 * q + 0] = v.x;
            xa[k][4 * q + 1] = v.y;
            xa[k][4 * q + 2] = v.z;
            xa[k][4 * q + 3] = v.w;
        }
    }
    if (M % 2) {
        const float4 *xp = reinterpret_cast<const float4 *>(x + 512 * (M / 2) + 8 * j);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const float4 v = xp[q];
            xb[4 * q + 0] = v.x;
            xb[4 * q + 1] = v.y;
            xb[4 * q + 2] = v.z;
            xb[4 * q + 3] = v.w;
        }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) rep4[i * kThreads + t] = make_float4(cbv[i], cbv[i], cbv[i], cbv[i]);
    __syncthreads();

    const float *cbl = reinterpret_cast<const float *>(rep4) + (lane & 31);
    float sp[kPasses];
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
        if (p == 0) {
#pragma unroll
            for (int q = kFirst; q < kPasses; ++q) {
                const int r = min(row0 + 2 * q, out - 1);
                load_row(c[q], w + size_t(r) * K, j);
            }
        }
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < M / 2; ++k) {
            const uint32_t dw[4] = {c[p].a[k].x, c[p].a[k].y, c[p].a[k].z, c[p].a[k].w};
#pragma unroll
            for (int d = 0; d < 4; ++d)
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const uint32_t e = (dw[d] >> (8 * b)) & 0xffu;
                    acc[b] += cbl[e * 32] * xa[k][4 * d + b];
                }
        }
        if (M % 2) {
            const uint32_t dw[2] = {c[p].b.x, c[p].b.y};
#pragma unroll
            for (int d = 0; d < 2; ++d)
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const uint32_t e = (dw[d] >> (8 * b)) & 0xffu;
                    acc[b] += cbl[e * 32] * xb[4 * d + b];
                }
        }
        sp[p] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    }
    // The eight rows' half-wave sums in one lane-exchange tree; lane j ends
    // with the row of pass half_wave_slot<8>(j), and lanes 4k store.
    const float s = ndl::half_wave_sum<kPasses>(sp, j);
    const int r = row0 + 2 * ndl::half_wave_slot<kPasses>(j);
    if ((j & 3) == 0 && r < out) y[r] = s;
}

// Any `in` (multiple of 16).  L lanes share a row, a wave's 64 / L rows of a pass
// take P passes; a step is U = 4 vectors of 16 codes a lane and row, and the
// next step's are issued before the current one's gathers.  L = 8, P = 2: 128
// contiguous bytes a row and load, eight loads of 16 bytes in flight.  The part
// step at a row's end goes first, its loads together with the first full step's:
// a vector past the end is read as the last one and left out of the sum.  The
// activations sit in LDS, the quads of a vector rotated by its index so that the
// lanes' reads of one quad fall on different banks; eight lanes a row read each
// once for two rows.
// Bound by HBM on stacks of wide rows, by filling the table for a tile on
// narrow ones.  Measured, MI355X, stacks of 300 MB, codes' GB/s (before: one
// load in flight a lane; 16 lanes a row): in = 64: 2289 (1122), 128: 3960
// (1671), 272: 3997 (1704), 528: 4989 (1869), 1040: 5000 (1922), 2048: 6087
// (1996), 4096: 5509 (1750).  Four lanes a row gain on 64 (2753) and lose
// elsewhere (4124 at 1040); 16 gain on 208 to 400 (12 % at most) and lose
// elsewhere (3701 at 4096).
// A problem of few rows has only its lanes to share the work, and rows past the
// end would repeat the last one's: 16 lanes a row up to 16 rows, a wave a row up
// to four.  us, eight lanes / so: 1 x 16 rows by 8000 25.3 / 9.3, by 16384 48.7 /
// 16.0; 2000 x 5 by 784 15.2 / 8.5; 1 x 3 by 16384 48.7 / 6.8 (16 lanes 15.8);
// 2000 x 4 by 4112 56.8 / 18.1 (24.7).
template <int L, int P>
__global__ __launch_bounds__(kThreads, 4) void cb8_gemv_any_kernel(
    const uint8_t *__restrict__ w, size_t w_stride, const float *__restrict__ cb,
    size_t cb_stride, const float *__restrict__ x, size_t x_stride, float *__restrict__ y,
    size_t y_stride, int out, int in)
{
    constexpr int U = 4, R = 64 / L;
    __shared__ float4 rep4[256 * 32 / 4];  // 32 KB
    extern __shared__ float4 xs4[];        // [in / 4]
    const size_t prob = blockIdx.y;
    w += prob * w_stride;
    cb += prob * cb_stride + size_t(blockIdx.x) * 256;
    x += prob * x_stride;
    y += prob * y_stride;
    const int t = threadIdx.x, lane = t & 63, j = lane & (L - 1);
    const int row0 = blockIdx.x * kTileRows + (t >> 6) * (R * P) + lane / L;
    const int nvec = in >> 4;

    const u32x4_t *wr[P];
#pragma unroll
    for (int p = 0; p < P; ++p)
        wr[p] = reinterpret_cast<const u32x4_t *>(w + size_t(min(row0 + R * p, out - 1)) * in);
    constexpr int kStep = U * L;
    const int tail = nvec / kStep * kStep;  // first vector of the part step
    u32x4_t cur[P][U], nxt[P][U];
    auto fetch = [&](u32x4_t (&c)[P][U], int v0) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int p = 0; p < P; ++p) c[p][u] = __builtin_nontemporal_load(wr[p] + v0 + u * L + j);
    };
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (tail + u * L < nvec) {
            const int v = min(tail + u * L + j, nvec - 1);
#pragma unroll
            for (int p = 0; p < P; ++p) nxt[p][u] = __builtin_nontemporal_load(wr[p] + v);
        }
    if (tail > 0) fetch(cur, 0);
    // float4 slot f4 = i*256 + t of the replica array holds entry f4 / 8.
    float cbv[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) cbv[i] = cb[(i * kThreads + t) >> 3];
    for (int f = t; f < in >> 2; f += kThreads) {
        const int v = f >> 2;
        xs4[4 * v + ((f ^ (v >> 2)) & 3)] = reinterpret_cast<const float4 *>(x)[f];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) rep4[i * kThreads + t] = make_float4(cbv[i], cbv[i], cbv[i], cbv[i]);
    __syncthreads();

    const float *cbl = reinterpret_cast<const float *>(rep4) + (lane & 31);
    float acc[P][8] = {};  // 8 L partial sums a row
    auto block = [&](const u32x4_t (&c)[P][U], int u, int v) {
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const float4 xq = xs4[4 * v + ((d ^ (v >> 2)) & 3)];
            const float xv[4] = {xq.x, xq.y, xq.z, xq.w};
#pragma unroll
            for (int p = 0; p < P; ++p)
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    acc[p][4 * (d & 1) + b] += cbl[((c[p][u][d] >> (8 * b)) & 0xffu) * 32] * xv[b];
        }
    };
    auto step = [&](const u32x4_t (&c)[P][U], int v0) {
#pragma unroll
        for (int u = 0; u < U; ++u) block(c, u, v0 + u * L + j);
    };
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (tail + u * L < nvec && tail + u * L + j < nvec) block(nxt, u, tail + u * L + j);
    for (int v0 = 0; v0 < tail; v0 += 2 * kStep) {
        if (v0 + kStep < tail) fetch(nxt, v0 + kStep);
        step(cur, v0);
        if (v0 + kStep >= tail) break;
        if (v0 + 2 * kStep < tail) fetch(cur, v0 + 2 * kStep);
        step(nxt, v0 + kStep);
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
        float s = ((acc[p][0] + acc[p][1]) + (acc[p][2] + acc[p][3])) +
                  ((acc[p][4] + acc[p][5]) + (acc[p][6] + acc[p][7]));
        if constexpr (L == 64) {
            s += ndl::wave_xor<32>(s);
            s += ndl::wave_xor<16>(s);
        }
        if constexpr (L >= 16) s += ndl::wave_xor<8>(s);
        s += ndl::wave_xor<4>(s);
        s += ndl::wave_xor<2>(s);
        s += ndl::wave_xor<1>(s);
        if (j == 0 && row0 + R * p < out) y[row0 + R * p] = s;
    }
}

// ---------------------------------------------------------------------------
// GEMM: Y[m][o] = sum_k bf16(X[m][k]) * bf16(cb[o/64][W[o][k]]), fp32 accumulate.
// ---------------------------------------------------------------------------
typedef __attribute__((__vector_size__(8 * sizeof(short)))) short bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4_t;

// fp32 to bf16, round to nearest even: gfx950's v_cvt_pk_bf16_f32 (two
// values an instruction).  It equals the integer form (u + 0x7fff + lsb) >> 16
// on every non-NaN input (a device sweep of all 2^32 patterns found no
// difference; test_gpu_cb8.py pins the ties through the GEMMs); NaNs stay NaN.
typedef __bf16 bf16x2_hw_t __attribute__((ext_vector_type(2)));

__device__ inline uint32_t f32x2_to_bf16x2_rne(float lo, float hi)
{
    const bf16x2_hw_t v = {static_cast<__bf16>(lo), static_cast<__bf16>(hi)};
    return __builtin_bit_cast(uint32_t, v);
}

__device__ inline unsigned short f32_to_bf16_rne(float f)
{
    return static_cast<unsigned short>(f32x2_to_bf16x2_rne(f, 0.0f));
}

constexpr int kGN = 64;     // columns sharing a codebook
constexpr int kLdsPad = 8;  // bf16 elements of padding per LDS row

// X (f32) to bf16, round to nearest even; problem blockIdx.y of a batch at
// element stride xs (input) and n (output).  A block converts kXRuns runs of
// 2048 elements, 8 per thread per run, all loads issued before the stores.
constexpr int kXRuns = 4;

__device__ inline uint4 pack_bf16x8(float4 a, float4 b)
{
    return make_uint4(f32x2_to_bf16x2_rne(a.x, a.y), f32x2_to_bf16x2_rne(a.z, a.w),
                      f32x2_to_bf16x2_rne(b.x, b.y), f32x2_to_bf16x2_rne(b.z, b.w));
}

__global__ __launch_bounds__(256) void x_to_bf16_kernel(const float *__restrict__ X, size_t xs,
                                                        unsigned short *__restrict__ Xb, size_t n)
{
    const float *src = X + blockIdx.y * xs;
    unsigned short *dst = Xb + blockIdx.y * n;
    const size_t base = size_t(blockIdx.x) * (2048 * kXRuns) + threadIdx.x * 8;
    if (base + 2048 * (kXRuns - 1) + 8 <= n) {
        float4 a[kXRuns], b[kXRuns];
#pragma unroll
        for (int r = 0; r < kXRuns; ++r) {
            a[r] = *reinterpret_cast<const float4 *>(src + base + 2048 * r);
            b[r] = *reinterpret_cast<const float4 *>(src + base + 2048 * r + 4);
        }
#pragma unroll
        for (int r = 0; r < kXRuns; ++r)
            *reinterpret_cast<uint4 *>(dst + base + 2048 * r) = pack_bf16x8(a[r], b[r]);
        return;
    }
    // a problem's last block: run by run, the ragged end element by element
    for (int r = 0; r < kXRuns; ++r) {
        const size_t i = base + 2048 * size_t(r);
        if (i >= n) return;
        if (i + 8 <= n) {
            const float4 a = *reinterpret_cast<const float4 *>(src + i);
            const float4 b = *reinterpret_cast<const float4 *>(src + i + 4);
            *reinterpret_cast<uint4 *>(dst + i) = pack_bf16x8(a, b);
        } else {
            for (size_t k = i; k < n; ++k) dst[k] = f32_to_bf16_rne(src[k]);
        }
    }
}

// Y[M][N] = X[M][K] . decode(W[N][K])^T, X already bf16, on 128x128 tiles (NB =
// 2): 4 waves of 64x64 (4x4 MFMA tiles each), K steps of 64, each thread staging
// half a row of A (32 bf16) and of B (32 codes); or 128x64 (NB = 1): 4 waves of
// 32x64, 16 codes a thread, the same order of K: the next step's are loaded into
// registers while the current step's MFMAs run from LDS.  The codebooks sit in
// LDS already rounded to bf16, so decoding a code is one LDS read.  With an odd
// number of 64-column groups the last 128-wide tile's second half repeats the
// last row and is not stored.
constexpr int kBM = 128, kBK = 64;

template <int NB>
__global__ __launch_bounds__(256) void cb8_gemm128_kernel(const unsigned short *__restrict__ Xb,
                                                          const uint8_t *__restrict__ W,
                                                          const float *__restrict__ cb,
                                                          float *__restrict__ Y, int M, int N,
                                                          int K, size_t ws, size_t cs, size_t ys)
{
    constexpr int BN = 64 * NB, MA = 2 * NB;  // columns; a wave's row tiles of 16
    constexpr int BC = 16 * NB;               // codes a thread stages
    __shared__ unsigned short cbh[NB][256];
    __shared__ __align__(16) unsigned short As[kBM][kBK + kLdsPad];
    __shared__ __align__(16) unsigned short Bs[BN][kBK + kLdsPad];

    Xb += blockIdx.z * size_t(M) * K;
    W += blockIdx.z * ws;
    cb += blockIdx.z * cs;
    Y += blockIdx.z * ys;

    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = t >> 6;
    const int n0 = blockIdx.x * BN;
    const int m0 = blockIdx.y * kBM;
    const int wm = NB == 2 ? (wave >> 1) * 64 : wave * 32;
    const int wn = NB == 2 ? (wave & 1) * 64 : 0;

    // the tile's codebooks, rounded to bf16
    cbh[0][t] = f32_to_bf16_rne(cb[size_t(n0 / 64) * 256 + t]);
    if constexpr (NB == 2) cbh[1][t] = f32_to_bf16_rne(cb[size_t(min(n0 / 64 + 1, N / 64 - 1)) * 256 + t]);

    floatx4_t acc[MA][4];
#pragma unroll
    for (int a = 0; a < MA; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};

    const int sr = t >> 1;          // staged row 0..127 of A
    const int sc = (t & 1) * 32;    // and columns sc..sc+31 of the K step
    const int br = NB == 2 ? sr : t >> 2, bc = NB == 2 ? sc : (t & 3) * 16;  // of B, BC columns
    const bool mrow = m0 + sr < M;
    const unsigned short *xrow = Xb + size_t(mrow ? m0 + sr : 0) * K;
    const uint8_t *wrow = W + size_t(min(n0 + br, N - 1)) * K;  // N is a multiple of 64
    const unsigned short *cbr = cbh[br >> 6];
    uint4 xa[4];
    uint2 wc[BC / 8];
    // a run of columns past K reads the one before it and is zeroed at the LDS
    // store: no load sits behind a branch
    auto load = [&](int k0) {
        const bool on = k0 + sc < K;
        const int kc = on ? k0 + sc : K - 32;
        const int kb = NB == 2 ? kc : (k0 + bc < K ? k0 + bc : K - BC);
#pragma unroll
        for (int q = 0; q < 4; ++q) xa[q] = *reinterpret_cast<const uint4 *>(xrow + kc + 8 * q);
#pragma unroll
        for (int q = 0; q < BC / 8; ++q) wc[q] = *reinterpret_cast<const uint2 *>(wrow + kb + 8 * q);
        return on;
    };
    auto store = [&](bool on, int k0) {
        const bool onb = NB == 2 ? on : k0 + bc < K;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *reinterpret_cast<uint4 *>(&As[sr][sc + 8 * q]) = on && mrow ? xa[q] : make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < BC / 8; ++q) {
            const uint32_t d[2] = {wc[q].x, wc[q].y};
            uint32_t h[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t lo = cbr[(d[e >> 1] >> (16 * (e & 1))) & 0xffu];
                const uint32_t hi = cbr[(d[e >> 1] >> (16 * (e & 1) + 8)) & 0xffu];
                h[e] = onb ? lo | (hi << 16) : 0u;
            }
            *reinterpret_cast<uint4 *>(&Bs[br][bc + 8 * q]) = make_uint4(h[0], h[1], h[2], h[3]);
        }
    };
    __syncthreads();
    bool on = load(0);
    const int r16 = lane & 15;
    const int kq = (lane >> 4) * 8;
    for (int k0 = 0; k0 < K; k0 += kBK) {
        store(on, k0);
        __syncthreads();
        if (k0 + kBK < K) on = load(k0 + kBK);
        const int steps = (K - k0 < kBK ? K - k0 : kBK) / 32;
        for (int kk = 0; kk < steps; ++kk) {
            bf16x8_t afrag[MA], bfrag[4];
#pragma unroll
            for (int a = 0; a < MA; ++a)
                afrag[a] = *reinterpret_cast<const bf16x8_t *>(&As[wm + a * 16 + r16][kk * 32 + kq]);
#pragma unroll
            for (int b = 0; b < 4; ++b)
                bfrag[b] = *reinterpret_cast<const bf16x8_t *>(&Bs[wn + b * 16 + r16][kk * 32 + kq]);
#pragma unroll
            for (int a = 0; a < MA; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(afrag[a], bfrag[b],
                                                                        acc[a][b], 0, 0, 0);
        }
        __syncthreads();
    }
    const int col = lane & 15;
    const int rb = (lane >> 4) * 4;
#pragma unroll
    for (int a = 0; a < MA; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = m0 + wm + a * 16 + rb + i;
                const int n = n0 + wn + b * 16 + col;
                if (m < M && n < N) Y[size_t(m) * N + n] = acc[a][b][i];
            }
}

// The same product on 256x256 tiles for launches with at least one tile per
// CU.  8 waves, two per SIMD, each a 64x128 output (4x8 MFMA 16x16x32 tiles);
// LDS holds two K steps of 64 so the next step is decoded while the current
// one is multiplied.  Waves 0-3 multiply first and then stage, waves 4-7
// stage first: the two waves sharing a SIMD are out of phase, so one keeps
// the MFMA pipe fed while the other waits on global loads and codebook
// gathers.  Loads read clamped, always valid addresses and are masked at the
// LDS store, so no load sits behind a branch.  Tiles are numbered so that each
// XCD (blocks are dealt round-robin to the 8 XCDs) owns a contiguous run,
// M tiles fastest: blocks sharing an X row block or a W column block meet in
// one L2.  Per output the K order is that of the 128x128 kernel, so the two
// agree bit for bit.
constexpr int kPM = 256, kPN = 256, kPK = 64;
constexpr int kPWM = 64, kPWN = 128;  // wave tile: waves 4 (M) x 2 (N)

__global__ __launch_bounds__(512) void cb8_gemm256_kernel(const float *__restrict__ Xf, size_t xs,
                                                          const uint8_t *__restrict__ W,
                                                          const float *__restrict__ cb,
                                                          float *__restrict__ Y, int M, int N,
                                                          int K, size_t ws, size_t cs, size_t ys,
                                                          int tiles_n, int tiles_m, int xcd_run)
{
    constexpr int TA = kPWM / 16, TB = kPWN / 16;
    constexpr int J = kPM / 64;  // staged 64-row slabs of A and of B
    __shared__ __align__(16) unsigned short As[2][kPM][kPK + kLdsPad];
    __shared__ __align__(16) unsigned short Bs[2][kPN][kPK + kLdsPad];
    __shared__ unsigned short cbh[kPN / 64][256];

    const int id = blockIdx.x;
    const int u = xcd_run ? (id % 8) * xcd_run + id / 8 : id;
    const int z = u / (tiles_n * tiles_m);
    const int m0 = (u % tiles_m) * kPM;
    const int n0 = ((u / tiles_m) % tiles_n) * kPN;
    Xf += z * xs;  // X stays fp32 in HBM; it is rounded to bf16 as it is staged
    W += z * ws;
    cb += z * cs;
    Y += z * ys;
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = t >> 6;
    const int wm = (wave & 3) * kPWM;
    const int wn = (wave >> 2) * kPWN;
    for (int i = t; i < kPN / 64 * 256; i += 512)
        cbh[i / 256][i % 256] = f32_to_bf16_rne(cb[size_t(n0 / 64 + i / 256) * 256 + i % 256]);

    floatx4_t acc[TA][TB];
#pragma unroll
    for (int a = 0; a < TA; ++a)
#pragma unroll
        for (int b = 0; b < TB; ++b) acc[a][b] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};

    const int r8 = t >> 3;       // staged row within a 64-row slab
    const int c8 = (t & 7) * 8;  // staged columns c8..c8+7 of the K step
    bool mok[J];
    const float *xp[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int m = m0 + r8 + 64 * j;
        mok[j] = m < M;
        xp[j] = Xf + size_t(m < M ? m : M - 1) * K + c8;
    }
    const uint8_t *wp = W + size_t(n0 + r8) * K + c8;  // N is a multiple of 256 here
    float4 xa[J][2];
    uint2 wc[J];
    bool on = true;
    auto load = [&](int k0) {
        on = k0 + c8 < K;
        // K is a multiple of 32: a run past K belongs to a final half step,
        // and the run 32 columns back is in range
        const int kc = on ? k0 : k0 - 32;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            xa[j][0] = *reinterpret_cast<const float4 *>(xp[j] + kc);
            xa[j][1] = *reinterpret_cast<const float4 *>(xp[j] + kc + 4);
        }
#pragma unroll
        for (int j = 0; j < J; ++j) wc[j] = *reinterpret_cast<const uint2 *>(wp + size_t(64 * j) * K + kc);
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int j = 0; j < J; ++j)
            *reinterpret_cast<uint4 *>(&As[buf][r8 + 64 * j][c8]) =
                on && mok[j] ? pack_bf16x8(xa[j][0], xa[j][1]) : make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const uint32_t d[2] = {wc[j].x, wc[j].y};
            uint32_t h[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t lo = cbh[j][(d[e >> 1] >> (16 * (e & 1))) & 0xffu];
                const uint32_t hi = cbh[j][(d[e >> 1] >> (16 * (e & 1) + 8)) & 0xffu];
                h[e] = on ? lo | (hi << 16) : 0u;
            }
            *reinterpret_cast<uint4 *>(&Bs[buf][r8 + 64 * j][c8]) = make_uint4(h[0], h[1], h[2], h[3]);
        }
    };
    const int r16 = lane & 15;
    const int kq = (lane >> 4) * 8;
    auto multiply = [&](int buf, int halves) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            if (kk < halves) {
                bf16x8_t af[TA], bfv[TB];
#pragma unroll
                for (int a = 0; a < TA; ++a)
                    af[a] = *reinterpret_cast<const bf16x8_t *>(&As[buf][wm + a * 16 + r16][kk * 32 + kq]);
#pragma unroll
                for (int b = 0; b < TB; ++b)
                    bfv[b] = *reinterpret_cast<const bf16x8_t *>(&Bs[buf][wn + b * 16 + r16][kk * 32 + kq]);
#pragma unroll
                for (int a = 0; a < TA; ++a)
#pragma unroll
                    for (int b = 0; b < TB; ++b)
                        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[a], bfv[b], acc[a][b], 0, 0, 0);
            }
        }
    };
    const int nk = (K + kPK - 1) / kPK;
    load(0);
    __syncthreads();  // codebooks in LDS
    store(0);
    load(nk > 1 ? kPK : 0);
    __syncthreads();
    const bool first = wave < 4;
    for (int i = 0; i < nk; ++i) {
        const int cur = i & 1;
        const int halves = (K - i * kPK < kPK ? K - i * kPK : kPK) / 32;
        // step i+1 into the other buffer (read last in step i-1, before the
        // barrier that ended it); step i+2's loads go out behind it.  Every
        // step stores and loads -- the last ones repeat the final step into a
        // buffer nothing reads -- so no load sits behind a branch and the
        // waits count the loads in flight exactly (a load behind a branch
        // makes the compiler wait for it at the join)
        const int kl = (i + 2 < nk ? i + 2 : nk - 1) * kPK;
        if (first) {
            multiply(cur, halves);
            store(cur ^ 1);
            load(kl);
        } else {
            store(cur ^ 1);
            load(kl);
            multiply(cur, halves);
        }
        __syncthreads();
    }
    const int col = lane & 15;
    const int rb = (lane >> 4) * 4;
#pragma unroll
    for (int a = 0; a < TA; ++a)
#pragma unroll
        for (int b = 0; b < TB; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = m0 + wm + a * 16 + rb + i;
                const int n = n0 + wn + b * 16 + col;
                if (m < M) Y[size_t(m) * N + n] = acc[a][b][i];
            }
}

// Tiles of 16 MT rows (all of them up to M = 64, e.g. the rows of 64 sessions
// at once) by 128 columns (two codebook groups), eight waves a block: each code
// feeds at most 64 rows, so the launch streams codes and the decode, not the
// MFMAs, sets the pace; the codes skip LDS.  Wave w takes columns 16 w ..
// 16 w + 15 through K steps of 128: lane (r16, q) loads codes 16q..16q+15 and
// 64+16q..64+16q+15 of row r16, the wave both halves of each 128-byte line
// (through the caches: with nontemporal loads the line came from memory twice,
// 43 us against 27 for 24 x 3 rows by 2624 x 2208), and decodes them through a
// lane-replicated codebook table (entry e, replica r in bank r: conflict-free
// gathers; both groups' bf16 in one word) straight into MFMA B fragments; a
// byte dot product forms an entry's address in one operation.  X is rounded to
// bf16 as it is staged in LDS, double buffered.  Codes and X are loaded two
// steps ahead.  Both operands use physical k 16q..16q+7 for the first MFMA of a
// half step and 16q+8..+15 for the second.  Without LINES a lane's codes come
// eight at a time, at 8q of each 32 k: for codes aligned to 8 bytes, and with
// the larger tiles' K order, bit for bit.  Past K (a last step of 32, 64 or
// 96), X is zero and the codes are a zero entry behind the codebook.
// Y is stored past the caches (64 problems of 64 rows by 6080 x 512: 92 -> 76
// us), whole lines through LDS (448 of 64 rows by 3072 x 768: 433 -> 416; half
// lines were written 1.2 times).
// Bound by LDS (gathers and X fragments) at 64 rows, by memory at few.
// Measured, MI355X, calls back to back (before: four waves of 32 columns, X
// rounded by a launch of its own; widths not a multiple of 128 in 64x64 tiles):
// 20 problems of 3072 x 768, 64 rows 23.9 -> 19.5 us, 16 rows 23.4 -> 12.6, 3
// rows 22.7 -> 12.1; 24 x 3 rows by 2624 x 2208 62.9 -> 25.0 (5.6 TB/s); 8 x 50
// by 768 x 3072 48.9 -> 30.5; 64 x 64 rows by 1024 x 3072 78.0 -> 59.0, by 3072
// x 768 63.3 -> 51.0, 448 of these, far past the caches, 409 -> 405.  32 columns
// and half the step a wave: 21.2 and 14.7 us for 20 problems of 64 and 16 rows.
// Up to a K of 128 (ONE) there is one step: nothing is loaded ahead, pieces past
// K are left out, and without a second buffer of X three blocks of 64 rows share
// a CU where two did.  us, 64x64 tiles before / with the steps' loop / so: 200 x
// 64 rows by 1984 x 32 26.7 / 33.2 / 21.0, 104 x 56 by 5312 x 96 37.6 / 43.5 /
// 30.7, 158 x 46 by 5440 x 128 71.9 / 76.7 / 47.0, 2000 x 1 by 192 x 128 24.4 /
// 28.5 / 15.5.
// Blocks of 512 threads a launch may have: HIP counts the threads of a dimension
// in 32 bits, and a launch of more leaves blocks out.
constexpr size_t kMaxBlocks512 = 0xffffffffu / 512;
constexpr int kRN = 128;          // output columns (N) per block: two codebook groups
constexpr int kRC = 128;          // K per step
constexpr int kRXS = kRC + 8;     // padded X row in LDS (bf16)

template <int MT, bool LINES, bool ONE>
__global__ __launch_bounds__(512, ONE ? 6 : 4) void cb8_gemm_rows_kernel(const float *__restrict__ X, size_t xstride,
                                                               const uint8_t *__restrict__ W,
                                                               const float *__restrict__ cb,
                                                               float *__restrict__ Y, int M, int N, int K,
                                                               size_t ws, size_t cs, size_t ys, int tiles_n,
                                                               int tiles_m, int xcd_run)
{
    __shared__ __align__(16) uint32_t tab[257 * 32];  // a zero entry behind the codebook
    __shared__ __align__(16) unsigned short xs[ONE ? 1 : 2][16 * MT * kRXS];
    __shared__ uint32_t one_vals[ONE ? 256 : 1];
    // the column tiles of one problem are consecutive in u and land on one
    // XCD (workgroups are dealt to the 8 XCDs round-robin), sharing X in L2
    const int id = blockIdx.x;
    const int u = xcd_run ? (id % 8) * xcd_run + id / 8 : id;
    const int z = u / (tiles_n * tiles_m), tm = u % tiles_m, tn = (u / tiles_m) % tiles_n;
    X += size_t(z) * xstride + size_t(tm) * (16 * MT) * K;
    Y += size_t(tm) * (16 * MT) * N;
    M = min(M - tm * (16 * MT), 16 * MT);
    W += z * ws;
    cb += z * cs;
    Y += z * ys;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int r16 = lane & 15, q = lane >> 4;
    const int n0 = tn * kRN, col = n0 + 16 * w + r16;
    const uint8_t *wp0 = W + size_t(min(col, N - 1)) * K;
    const int k0 = LINES ? 16 * q : 8 * q;
    const int nc = (K + kRC - 1) / kRC;
    // every step issues the same loads (addresses clamped), so the waits
    // count them exactly
    u32x4_t cw[2][2];
    auto cload = [&](int slot, int c) {
        if constexpr (LINES) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                // the second read of a line is its last
                const u32x4_t *p = reinterpret_cast<const u32x4_t *>(wp0 + min(c * kRC + 64 * h + k0, K - 16));
                cw[slot][h] = h ? __builtin_nontemporal_load(p) : *p;
            }
        } else {
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                const u32x2_t v = *reinterpret_cast<const u32x2_t *>(wp0 + min(c * kRC + 32 * h + k0, K - 8));
                cw[slot][h >> 1][2 * (h & 1)] = v.x;
                cw[slot][h >> 1][2 * (h & 1) + 1] = v.y;
            }
        }
    };
    // X of step c: 16 MT rows x 128, four columns a thread and piece
    float4 xr[MT];
    const int xrow = t >> 5, xcol = (t & 31) * 4;
    auto xload = [&](int c) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
            xr[i] = *reinterpret_cast<const float4 *>(X + size_t(min(xrow + 16 * i, M - 1)) * K +
                                                            min(c * kRC + xcol, K - 4));
    };
    auto xstore = [&](int buf, int c) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const float4 v = xr[i];
            uint2 h = make_uint2(f32x2_to_bf16x2_rne(v.x, v.y), f32x2_to_bf16x2_rne(v.z, v.w));
            if (xrow + 16 * i >= M || c * kRC + xcol >= K) h = make_uint2(0, 0);
            *reinterpret_cast<uint2 *>(&xs[buf][(xrow + 16 * i) * kRXS + xcol]) = h;
        }
    };
    xload(0);
    cload(0, 0);
    if constexpr (!ONE) cload(1, 1);
    {
        // the table, through a staging row (in xs[1] where there is one) so
        // every write is conflict-free: word e of the row, then 4 x 16 bytes a
        // thread
        uint32_t *vals = ONE ? one_vals : reinterpret_cast<uint32_t *>(&xs[ONE ? 0 : 1][0]);
        const int ng = N / 64 - 1;
        if (t < 256)
            vals[t] = f32_to_bf16_rne(cb[size_t(n0 / 64) * 256 + t]) |
                      (uint32_t(f32_to_bf16_rne(cb[size_t(min(n0 / 64 + 1, ng)) * 256 + t])) << 16);
        __syncthreads();
        uint4 *t4 = reinterpret_cast<uint4 *>(tab);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t v = vals[(i * 512 + t) >> 3];
            t4[i * 512 + t] = make_uint4(v, v, v, v);
        }
    }
    if (t < 32) tab[256 * 32 + t] = 0;
    xstore(0, 0);
    if constexpr (!ONE) xload(1);
    __syncthreads();
    // waves 0-3 hold rows of the first group (low halves), 4-7 the second
    const uint32_t sel = w >= 4 ? 0x07060302u : 0x05040100u;
    typedef __attribute__((address_space(3))) uint32_t *lds_u32;
    const uint32_t base = uint32_t(reinterpret_cast<uintptr_t>((lds_u32)(tab + (lane & 31))));
    floatx4_t acc[MT];
#pragma unroll
    for (int a = 0; a < MT; ++a) acc[a] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};
    // one dot product of bytes makes an entry's address; codes past the end
    // are the zero entry
    auto decode = [&](uint32_t d0, uint32_t d1, bool in) {
        const uint32_t at = in ? base : base + 256 * 128;
        const uint32_t dw[2] = {in ? d0 : 0u, in ? d1 : 0u};
        uint32_t h[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t v0 = *(lds_u32)(uintptr_t(__builtin_amdgcn_udot4(dw[k >> 1], 0x80u << (16 * (k & 1)), at, false)));
            const uint32_t v1 = *(lds_u32)(uintptr_t(__builtin_amdgcn_udot4(dw[k >> 1], 0x8000u << (16 * (k & 1)), at, false)));
            h[k] = __builtin_amdgcn_perm(v1, v0, sel);
        }
        return __builtin_bit_cast(bf16x8_t, make_uint4(h[0], h[1], h[2], h[3]));
    };
    // piece h of a step, eight codes: where its k start for this lane
    auto piece = [&](int h) { return LINES ? 64 * (h >> 1) + 8 * (h & 1) + k0 : 32 * h + k0; };
    if constexpr (ONE) {
        // pieces wholly past K are left out
#pragma unroll
        for (int h = 0; h < 4; ++h)
            if ((LINES ? 64 * (h >> 1) : 32 * h) < K) {
                const bf16x8_t b = decode(cw[0][h >> 1][2 * (h & 1)], cw[0][h >> 1][2 * (h & 1) + 1], piece(h) < K);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        *reinterpret_cast<const bf16x8_t *>(&xs[0][(16 * mt + r16) * kRXS + piece(h)]), b, acc[mt], 0, 0, 0);
            }
        __syncthreads();
    }
    for (int c0 = 0; !ONE && c0 < nc; c0 += 2) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int c = c0 + s;
            if (c < nc) {
                // X of step c + 1 into the buffer that step c - 1 read
                xstore(ONE ? 0 : s ^ 1, c + 1);
                xload(c + 2);
                bf16x8_t b[4];
#pragma unroll
                for (int h = 0; h < 4; ++h)
                    b[h] = decode(cw[s][h >> 1][2 * (h & 1)], cw[s][h >> 1][2 * (h & 1) + 1],
                                  c * kRC + piece(h) < K);
                cload(s, c + 2);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int h = 0; h < 4; ++h)
                        acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            *reinterpret_cast<const bf16x8_t *>(&xs[ONE ? 0 : s][(16 * mt + r16) * kRXS + piece(h)]), b[h],
                            acc[mt], 0, 0, 0);
                __syncthreads();
            }
        }
    }
    // the tile through the table's LDS, so that whole lines are stored: columns
    // of 16 exchanged by row so that a wave's writes fall on all banks
    float *yt = reinterpret_cast<float *>(tab);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            yt[(16 * mt + 4 * q + i) * kRN + ((16 * w + r16) ^ (16 * q))] = acc[mt][i];
    __syncthreads();
    typedef float f32x4_any_t __attribute__((ext_vector_type(4), aligned(4)));  // Y is aligned as floats are
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int m = xrow + 16 * i;
        const f32x4_any_t v = *reinterpret_cast<const f32x4_any_t *>(yt + m * kRN + (xcol ^ (16 * ((m >> 2) & 3))));
        if (m < M && n0 + xcol < N)
            __builtin_nontemporal_store(v, reinterpret_cast<f32x4_any_t *>(Y + size_t(m) * N + n0 + xcol));
    }
}

int launch_gemv(nd_ctx *ctx, size_t count, const uint8_t *w, size_t w_stride, const float *cb,
                size_t cb_stride, const float *x, size_t x_stride, float *y, size_t y_stride,
                size_t out, size_t in)
{
    ND_REQUIRE(w && cb && x && y, "null buffer");
    ND_REQUIRE(out > 0 && in > 0, "empty shape %zux%zu", out, in);
    ND_REQUIRE(in % 16 == 0, "in (%zu) must be a multiple of 16", in);
    ND_REQUIRE(out <= (size_t(1) << 30) && in <= (size_t(1) << 24), "shape too large");
    ND_REQUIRE(count >= 1 && count <= 65535, "count %zu out of range 1..65535", count);
    ND_REQUIRE((reinterpret_cast<uintptr_t>(w) & 15) == 0 && w_stride % 16 == 0,
               "codes must be 16-byte aligned");
    ND_REQUIRE((reinterpret_cast<uintptr_t>(x) & 15) == 0 && x_stride % 4 == 0,
               "activations must be 16-byte aligned");
    const int tiles = static_cast<int>((out + kTileRows - 1) / kTileRows);
    dim3 grid(tiles, static_cast<unsigned>(count));
    const bool fast = in % 256 == 0 && in <= 1024 && (reinterpret_cast<uintptr_t>(x) & 15) == 0 &&
                      x_stride % 4 == 0;
#define ND_GEMV(MM)                                                                          \
    hipLaunchKernelGGL((cb8_gemv_kernel<MM>), grid, dim3(kThreads), 0, ctx->stream, w, w_stride, \
                       cb, cb_stride, x, x_stride, y, y_stride, int(out))
    if (fast) {
        switch (in / 256) {
        case 1: ND_GEMV(1); break;
        case 2: ND_GEMV(2); break;
        case 3: ND_GEMV(3); break;
        default: ND_GEMV(4); break;
        }
    } else {
        ND_REQUIRE(in * sizeof(float) <= 64 * 1024, "in (%zu) too large", in);
#define ND_GEMV_ANY(L, P)                                                                             \
    hipLaunchKernelGGL((cb8_gemv_any_kernel<L, P>), grid, dim3(kThreads), in * sizeof(float), ctx->stream, w, \
                       w_stride, cb, cb_stride, x, x_stride, y, y_stride, int(out), int(in))
        if (out <= 4)
            ND_GEMV_ANY(64, 1);
        else if (out <= 16)
            ND_GEMV_ANY(16, 1);
        else
            ND_GEMV_ANY(8, 2);
#undef ND_GEMV_ANY
    }
#undef ND_GEMV
    return nd::check_launch("cb8_gemv");
}

}  // namespace

extern "C" {

int nd_cb8_gemv(nd_ctx *ctx, const uint8_t *w, const float *cb, const float *x, float *y,
                size_t out, size_t in)
{
    ND_ENTER(ctx);
    return launch_gemv(ctx, 1, w, 0, cb, 0, x, 0, y, 0, out, in);
}

int nd_cb8_gemv_batched(nd_ctx *ctx, size_t count, const uint8_t *w, size_t w_stride,
                        const float *cb, size_t cb_stride, const float *x, size_t x_stride,
                        float *y, size_t y_stride, size_t out, size_t in)
{
    ND_ENTER(ctx);
    return launch_gemv(ctx, count, w, w_stride, cb, cb_stride, x, x_stride, y, y_stride, out, in);
}

int nd_cb8_gemm_batched(nd_ctx *ctx, size_t count, const float *x, size_t x_stride,
                        const uint8_t *w, size_t w_stride, const float *cb, size_t cb_stride,
                        float *y, size_t y_stride, size_t m, size_t out, size_t in)
{
    ND_ENTER(ctx);
    if (count == 0) return ND_OK;
    ND_REQUIRE(x && w && cb && y, "null buffer");
    ND_REQUIRE(m > 0 && out > 0 && in > 0, "empty shape");
    ND_REQUIRE(count <= 65535, "count %zu above 65535", count);
    ND_REQUIRE(out % kGN == 0, "out (%zu) must be a multiple of %d", out, kGN);
    ND_REQUIRE(in % 32 == 0, "in (%zu) must be a multiple of 32", in);
    ND_REQUIRE(m <= (size_t(1) << 24) && out <= (size_t(1) << 24) && in <= (size_t(1) << 24),
               "shape too large");
    ND_REQUIRE((reinterpret_cast<uintptr_t>(x) & 15) == 0 && (reinterpret_cast<uintptr_t>(w) & 7) == 0 &&
                   x_stride % 4 == 0 && w_stride % 8 == 0,
               "x must be 16-byte and w 8-byte aligned, problem by problem");
    const size_t big_tiles = (out / kPN) * ((m + kPM - 1) / kPM) * count;
    const size_t cus = size_t(ctx->num_cus > 0 ? ctx->num_cus : 256);
    // 64-row tiles where m has no more, and where two a CU hold them all: a
    // launch that does not fill the chip waits for one tile's steps, which are
    // shorter there (us, rows / 128x128 tiles: 192 tiles of 1 x 512 by 3072 x
    // 768 14.0 / 22.1, 384 of 8 x 500 by 768 x 768 23.9 / 29.2, 512 of 4 x 1000
    // by 1024 x 256 14.5 / 15.6, 720 of 6 x 300 by 3072 x 768 34.7 / 33.1, 960
    // of 20 x 80 by 3072 x 768 46.2 / 32.7).  Whole lines of codes need them
    // 16-byte aligned.  Above 64 rows the K order is the larger tiles', so a
    // problem's bits do not depend on how many share its launch.
    const size_t row_tiles_m = (m + 63) / 64;
    const size_t row_tiles = ((out + kRN - 1) / kRN) * row_tiles_m * count;
    const bool lines = m <= 64 && (reinterpret_cast<uintptr_t>(w) & 15) == 0 && w_stride % 16 == 0;
    const bool use_rows = m <= 64 || row_tiles <= 2 * cus;
    const bool use_256 = !use_rows && m >= 96 && out % kPN == 0 && big_tiles >= cus && big_tiles <= kMaxBlocks512;
    // X to bf16 once per call, into the context workspace, for the kernels
    // that stage bf16 X; the 256x256 and the row kernel round fp32 X as they
    // stage it
    const size_t mk = m * in;
    unsigned short *xb = nullptr;
    if (!use_256 && !use_rows) {
        void *wsp = nullptr;
        if (int rc = nd::workspace(ctx, count * mk * sizeof(unsigned short), &wsp)) return rc;
        xb = static_cast<unsigned short *>(wsp);
        hipLaunchKernelGGL(x_to_bf16_kernel, dim3(unsigned((mk + 2048 * kXRuns - 1) / (2048 * kXRuns)), unsigned(count)),
                           dim3(256), 0, ctx->stream, x, x_stride, xb, mk);
        if (int rc = nd::check_launch("x_to_bf16")) return rc;
    }
    if (use_rows) {
        // one launch, or as many problems a launch as its grid may hold (a
        // problem has 2^17 tiles at most)
        const size_t tiles_n = (out + kRN - 1) / kRN, tiles = tiles_n * row_tiles_m;
        const size_t most = kMaxBlocks512 / tiles;
        for (size_t z0 = 0; z0 < count; z0 += most) {
            const size_t blocks = (count - z0 < most ? count - z0 : most) * tiles;
            const int run = blocks % 8 == 0 ? int(blocks / 8) : 0;
#define ND_GEMM_ROWS(MT, LINES)              \
    if (in <= size_t(kRC))                   \
        ND_GEMM_ROWS_ONE(MT, LINES, true);   \
    else                                     \
        ND_GEMM_ROWS_ONE(MT, LINES, false)
#define ND_GEMM_ROWS_ONE(MT, LINES, ONE)                                                                \
    hipLaunchKernelGGL((cb8_gemm_rows_kernel<MT, LINES, ONE>), dim3(unsigned(blocks)), dim3(512), 0, ctx->stream, \
                       x + z0 * x_stride, x_stride, w + z0 * w_stride, cb + z0 * cb_stride,             \
                       y + z0 * y_stride, int(m), int(out), int(in), w_stride, cb_stride, y_stride,     \
                       int(tiles_n), int(row_tiles_m), run)
            if (!lines) {
                ND_GEMM_ROWS(4, false);
            } else if (m <= 16) {
                ND_GEMM_ROWS(1, true);
            } else if (m <= 32) {
                ND_GEMM_ROWS(2, true);
            } else {
                ND_GEMM_ROWS(4, true);
            }
            if (int rc = nd::check_launch("cb8_gemm")) return rc;
        }
#undef ND_GEMM_ROWS
#undef ND_GEMM_ROWS_ONE
    } else if (use_256) {
        // at least one 256x256 tile per CU: below that the 128x128 tiles fill
        // the chip better
        const int run = big_tiles % 8 == 0 ? int(big_tiles / 8) : 0;
        hipLaunchKernelGGL(cb8_gemm256_kernel, dim3(unsigned(big_tiles)), dim3(512), 0, ctx->stream, x,
                           x_stride, w, cb, y, int(m), int(out), int(in), w_stride, cb_stride, y_stride,
                           int(out / kPN), int((m + kPM - 1) / kPM), run);
    } else {
#define ND_GEMM128(NB)                                                                                 \
    hipLaunchKernelGGL(cb8_gemm128_kernel<NB>,                                                           \
                       dim3(unsigned((out + 64 * NB - 1) / (64 * NB)), unsigned((m + kBM - 1) / kBM), unsigned(count)), \
                       dim3(256), 0, ctx->stream, xb, w, cb, y, int(m), int(out), int(in), w_stride, cb_stride, y_stride)
        // 128x64 tiles for a small odd number of 64-column groups where half of
        // the 128x128 tiles' area or more would be idle (us, 128x128 / 128x64: 200
        // x 130 rows by 64 x 768 43.0 / 36.7, 46 x 2000 by 64 x 96 20.9 / 19.0,
        // 250 x 130 by 192 x 96 23.9 / 19.3, 416 x 130 by 448 x 256 83.1 / 71.8);
        // with less idle, or more columns, the wider tile is as fast or faster
        // (49 x 130 by 4032 x 1408 240 / 287, 448 columns by 500 rows 1.09)
        const size_t bm = (m + kBM - 1) / kBM * kBM, bn = (out + 127) / 128 * 128;
        if (out % 128 != 0 && out <= 448 && 2 * m * out <= bm * bn)
            ND_GEMM128(1);
        else
            ND_GEMM128(2);
#undef ND_GEMM128
    }
    return nd::check_launch("cb8_gemm");
}

int nd_cb8_gemm(nd_ctx *ctx, const float *x, const uint8_t *w, const float *cb, float *y,
                size_t m, size_t out, size_t in)
{
    return nd_cb8_gemm_batched(ctx, 1, x, 0, w, 0, cb, 0, y, 0, m, out, in);
}

}  // extern "C"
