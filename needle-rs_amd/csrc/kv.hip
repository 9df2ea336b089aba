// int8 KV cache: quantise-on-append and decode attention that reads the int8
// cache directly (crates/needle-core/src/v3/cache.rs, v3/attention.rs).
//
// Quantisation is bit-exact with quant_scale/quant_into (cache.rs:80-104):
// absmax (order-free), scale = absmax / 127 with an IEEE divide,
// inv = 1 / scale, q = clamp(roundf(x * inv), -128, 127), roundf being
// round-half-away-from-zero as libm::roundf.  One wave per head vector.
//
// Attention (attend_step over Int8View, attention.rs:300-377) reads the int8
// cache directly, in chunks with an online softmax (flash decoding).  One query
// head a kv head: attn_i8_kernel, a workgroup a (query, kv head).  Two or more,
// and the rows of a prompt over one cache: attn_mm_kernel, on the matrix cores,
// a wave 16 or 32 (row, head) columns of a kv head, so its int8 rows are read
// once for all of them.  The span is split across workgroups, with a merge
// pass, only when there are too few of them to fill the GPU (batch-1 decode).
#include "nd_internal.h"
#include "nd_kv_internal.h"

#include <cmath>
#include <mutex>

// Split-K partials of nd_attend_step_i8_noalloc: one fixed device array per
// GPU (every device the library runs on holds its copy until the process
// ends).  Host code never passes `scratch` itself to a kernel: its name is a
// host-side stand-in, and the device address comes from hipGetSymbolAddress
// once per device (nd::noalloc_setup, called when a context is created; if
// it fails there, the context is still created and this entry point reports
// the missing address).
static constexpr size_t kNoAllocScratchFloats = size_t(1) << 20;  // 4 MiB
static __device__ __align__(256) float scratch[kNoAllocScratchFloats];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
float *g_scratch[kMaxDevices] = {};
}  // namespace

namespace nd {

int noalloc_setup(int device)
{
    if (device < 0 || device >= kMaxDevices)
        return fail(ND_ERR_ARG, "device %d beyond the %d the no-allocation scratch covers", device,
                    kMaxDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch[device]) return ND_OK;
    void *p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
    if (!p) return fail(ND_ERR_HIP, "hipGetSymbolAddress(scratch) gave a null address");
    g_scratch[device] = static_cast<float *>(p);
    return ND_OK;
}

}  // namespace nd

namespace {

using namespace ndkv;

constexpr int kThreads = 256;

// fake_quant_vec over rows (cache.rs:68-73); one wave per row.
__global__ __launch_bounds__(kThreads) void fake_quant_kernel(float *__restrict__ x, size_t rows,
                                                             int dim)
{
    const size_t r = size_t(blockIdx.x) * (kThreads / 64) + (threadIdx.x >> 6);
    if (r >= rows) return;
    float *v = x + r * dim;
    float scale, inv;
    quant_scale_wave(v, dim, scale, inv);
    for (int i = threadIdx.x & 63; i < dim; i += 64) v[i] = quant_code(v[i], inv) * scale;
}

// quantize_rows (cache.rs:113-122); one wave per row.
__global__ __launch_bounds__(kThreads) void quantize_rows_kernel(const float *__restrict__ x,
                                                                size_t rows, int dim,
                                                                int8_t *__restrict__ q,
                                                                float *__restrict__ scales)
{
    const size_t r = size_t(blockIdx.x) * (kThreads / 64) + (threadIdx.x >> 6);
    if (r >= rows) return;
    const float *v = x + r * dim;
    float scale, inv;
    quant_scale_wave(v, dim, scale, inv);
    for (int i = threadIdx.x & 63; i < dim; i += 64) q[r * dim + i] = int8_t(quant_code(v[i], inv));
    if ((threadIdx.x & 63) == 0) scales[r] = scale;
}


// write_kv (cache.rs:346-379): wave w of block (i, h) quantises K (w=0) or
// V (w=1) of kv head h for row i into slot pos[i] % cap.
__global__ __launch_bounds__(128) void kv_write_kernel(Geom g, uint8_t *__restrict__ kv,
                                                      size_t kv_stride,
                                                      const int32_t *__restrict__ pos,
                                                      const float *__restrict__ k,
                                                      const float *__restrict__ v)
{
    const size_t i = blockIdx.x;
    const int h = blockIdx.y;
    const int which = threadIdx.x >> 6;
    const int p = pos[i];
    if (p < 0) return;
    const int slot = p % g.cap;
    uint8_t *blk = kv + i * kv_stride;
    const int dim = which ? g.VD : g.QK;
    const float *src = which ? v + i * size_t(g.KVH) * g.VD + size_t(h) * g.VD
                             : k + i * size_t(g.KVH) * g.QK + size_t(h) * g.QK;
    int8_t *dst = reinterpret_cast<int8_t *>(blk + (which ? g.v_off : 0)) +
                  (size_t(h) * g.cap + slot) * dim;
    float *sc = reinterpret_cast<float *>(blk + (which ? g.vs_off : g.ks_off)) + size_t(h) * g.cap + slot;
    float scale, inv;
    quant_scale_wave(src, dim, scale, inv);
    for (int e = threadIdx.x & 63; e < dim; e += 64) dst[e] = int8_t(quant_code(src[e], inv));
    if ((threadIdx.x & 63) == 0) *sc = scale;
}

// write_kv with KvPrecision::F32 (cache.rs:359-362): block (i, h) copies kv
// head h's K and V of row i into slot pos[i] % cap of the f32 block.
__global__ __launch_bounds__(64) void kv_write_f32_kernel(Geom g, uint8_t *__restrict__ kv,
                                                          size_t kv_stride,
                                                          const int32_t *__restrict__ pos,
                                                          const float *__restrict__ k,
                                                          const float *__restrict__ v)
{
    const size_t i = blockIdx.x;
    const int h = blockIdx.y;
    const int p = pos[i];
    if (p < 0) return;
    const int slot = p % g.cap;
    uint8_t *blk = kv + i * kv_stride;
    const float *ks = k + (i * size_t(g.KVH) + h) * g.QK;
    const float *vs = v + (i * size_t(g.KVH) + h) * g.VD;
    float *kd = reinterpret_cast<float *>(blk) + (size_t(h) * g.cap + slot) * g.QK;
    float *vd = reinterpret_cast<float *>(blk + g.v_off) + (size_t(h) * g.cap + slot) * g.VD;
    for (int e = threadIdx.x; e < g.QK; e += 64) kd[e] = ks[e];
    for (int e = threadIdx.x; e < g.VD; e += 64) vd[e] = vs[e];
}

// ---------------------------------------------------------------------------
// Decode attention over the int8 ring with one query head a kv head,
// flash-decoding style: the HBM stream (grouped heads share a K/V row and
// take the matrix-core kernel below).
//
// Block = (query i, kv head g, split s).  It walks its share of the span in
// chunks of CH positions with an online softmax (running max m, running sum
// l, accumulator rescaled by exp(m_old - m_new)), so one block can cover a
// whole span and no merge is needed when sessions x kv heads fill the GPU.
// Register pipeline: a chunk's K and V are already in registers when it
// starts; the next chunk's K loads are issued as soon as the scores are
// done, and its V loads as soon as the value pass is done.
//   K: KL = qk/16 lanes per position, one 16-byte int8 vector each, the
//      lane's 16-wide slice of the query head in registers.
//   V: VL = vd/16 lanes per position, 16 bytes each, 16 accumulators a lane.
// Scores, weights and block reductions go through LDS.
template <int QK, int VD>
struct AttnShape {
    static constexpr int KL = QK / 16;
    static constexpr int KPP = kThreads / KL;                 // positions per K pass
    static constexpr int VL = VD / 16;
    static constexpr int VPP = kThreads / VL;                 // positions per V pass
    // positions per chunk: 256 keeps the registers at 119 (four waves a
    // SIMD) and two chunks of a 512-long span in flight; 512 took 157
    // (three), and at 12 heads x 64 measured 5.37 / 5.96 / 5.96 TB/s at ctx
    // 512 / 2048 / 8192 against 5.69 / 6.32 / 6.34 with 256 (192: 5.10 /
    // 5.83 / 5.91; 384: 4.43 / 5.47 / 5.73)
    static constexpr int CH = 256;
    static constexpr int KP = (CH + KPP - 1) / KPP;           // K passes per chunk
    // KL a power of two (qk 16 .. 256) and one pass per lane of a position:
    // the KL partial dots meet through DPP in registers, no LDS and no
    // barrier.  qk 48 (three lanes a position) sums them in LDS
    static constexpr bool kLaneSums = (KL & (KL - 1)) == 0 && KL <= 16 && KP == KL && KPP * KL == kThreads;
    static constexpr int VP = CH / VPP;                       // V passes per chunk
};

__device__ inline float i8_at(uint32_t dw, int b) { return float(int32_t(dw << (24 - 8 * b)) >> 24); }

template <int QK, int VD>
__global__ __launch_bounds__(kThreads) void attn_i8_kernel(
    Geom g, const uint8_t *__restrict__ kv, size_t kv_stride, const int32_t *__restrict__ lo_a,
    const int32_t *__restrict__ hi_a, const float *__restrict__ q, float scale, int quant_query,
    int splits, float *__restrict__ out, float *__restrict__ part_o, float *__restrict__ part_ml)
{
    using S = AttnShape<QK, VD>;
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    constexpr int CH = S::CH, NW = kThreads / 64;
    __shared__ float qs[QK];
    __shared__ float sp[CH * S::KL];  // lane partial dots
    __shared__ float wsh[CH];         // scores, then weights
    __shared__ float red[NW];
    __shared__ float vred[NW][VD];

    const size_t qi = blockIdx.z;
    const int kvh = blockIdx.y;
    const int split = blockIdx.x;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;

    const int lo = lo_a[qi], hi = hi_a[qi];
    const int span = hi - lo + 1;
    const bool bad = lo < 0 || span < 1 || span > g.cap;
    const int nch = bad ? 0 : (span + CH - 1) / CH;
    // nch <= 2^16 chunks and splits <= 2^15: the products fit in 32 bits
    const int c_begin = int(uint32_t(nch) * uint32_t(split) / uint32_t(splits));
    const int c_end = int(uint32_t(nch) * uint32_t(split + 1) / uint32_t(splits));
    // a span is no longer than the ring: positions wrap at most once
    const int slo = bad ? 0 : lo % g.cap;
    auto slot_of = [&](int pc) {
        const int s = slo + pc;
        return s >= g.cap ? s - g.cap : s;
    };

    const uint8_t *blk = kv + qi * kv_stride;
    const int8_t *kb = reinterpret_cast<const int8_t *>(blk) + size_t(kvh) * g.cap * QK;
    const int8_t *vb = reinterpret_cast<const int8_t *>(blk + g.v_off) + size_t(kvh) * g.cap * VD;
    const float *ksb = reinterpret_cast<const float *>(blk + g.ks_off) + size_t(kvh) * g.cap;
    const float *vsb = reinterpret_cast<const float *>(blk + g.vs_off) + size_t(kvh) * g.cap;

    // The query head (fake-quantised on request).
    const float *qg = q + qi * size_t(g.H) * QK + size_t(kvh) * QK;
    for (int e = t; e < QK; e += kThreads) qs[e] = qg[e];
    __syncthreads();
    if (quant_query) {
        if (wave == 0) {
            float sc, inv;
            quant_scale_wave(qs, QK, sc, inv);
            for (int e = lane; e < QK; e += 64) qs[e] = quant_code(qs[e], inv) * sc;
        }
        __syncthreads();
    }
    const int ksub = t % S::KL;
    const int kpos = t / S::KL;  // position within a K pass
    const bool kact = t < S::KPP * S::KL;
    float qr[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) qr[e] = qs[ksub * 16 + e];
    const int vsub = t % S::VL;
    const int vpos = t / S::VL;

    u4 kr[S::KP], vr[S::VP];
    auto load_k = [&](int c) {
#pragma unroll
        for (int p = 0; p < S::KP; ++p) {
            const int pl = p * S::KPP + kpos;
            const int pc = min(c * CH + pl, span - 1);  // clamp: read a valid slot
            const int slot = slot_of(pc);
            kr[p] = __builtin_nontemporal_load(reinterpret_cast<const u4 *>(kb + size_t(slot) * QK) + ksub);
        }
    };
    auto load_v = [&](int c) {
#pragma unroll
        for (int p = 0; p < S::VP; ++p) {
            const int pc = min(c * CH + p * S::VPP + vpos, span - 1);
            const int slot = slot_of(pc);
            vr[p] = __builtin_nontemporal_load(reinterpret_cast<const u4 *>(vb + size_t(slot) * VD) + vsub);
        }
    };
    if (c_begin < c_end) {
        load_k(c_begin);
        load_v(c_begin);
    }

    float m_run = -INFINITY, l_loc = 0.0f, acc[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.0f;

    // a lane's partial dot of K pass p
    auto dot16 = [&](int p) {
        const uint32_t dw[4] = {kr[p].x, kr[p].y, kr[p].z, kr[p].w};
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int e = 0; e < 16; e += 2) {
            a0 += qr[e] * i8_at(dw[e >> 2], e & 3);
            a1 += qr[e + 1] * i8_at(dw[e >> 2], (e & 3) + 1);
        }
        return a0 + a1;
    };
    for (int c = c_begin; c < c_end; ++c) {
        const int n = min(CH, span - c * CH);
        float cmax = -INFINITY;
        // the position this lane scores, its score and V scale (lane sums)
        const int own = ksub * S::KPP + kpos;
        float own_sc = 0.0f, own_vs = 0.0f;
        if constexpr (S::kLaneSums) {
            // ---- scores: lane partial dots summed across the position's KL
            // lanes by DPP; lane ksub keeps pass ksub's position, and its
            // K and V scales are requested before the dots ----
            const int oslot = slot_of(c * CH + min(own, n - 1));
            const float ks = ksb[oslot];
            own_vs = vsb[oslot];
            float dot = 0.0f;
#pragma unroll
            for (int p = 0; p < S::KP; ++p) {
                const float v = ndl::group_sum<S::KL>(dot16(p));
                dot = ksub == p ? v : dot;
            }
            if (c + 1 < c_end) load_k(c + 1);  // lands during softmax and values
            own_sc = (dot * ks) * scale;
            if (own < n) cmax = own_sc;
        } else {
            // ---- scores: lane partial dots, then per position ----
#pragma unroll
            for (int p = 0; p < S::KP; ++p) {
                const int pl = p * S::KPP + kpos;
                if (kact && pl < CH) sp[pl * S::KL + ksub] = dot16(p);
            }
            if (c + 1 < c_end) load_k(c + 1);  // lands during softmax and values
            __syncthreads();
            for (int pl = t; pl < n; pl += kThreads) {
                const int slot = slot_of(c * CH + pl);
                float a = 0.0f;
#pragma unroll
                for (int s2 = 0; s2 < S::KL; ++s2) a += sp[pl * S::KL + s2];
                const float sc = (a * ksb[slot]) * scale;
                wsh[pl] = sc;
                cmax = fmaxf(cmax, sc);
            }
        }
        const float wm = wave_max(cmax);
        if (lane == 0) red[wave] = wm;
        __syncthreads();
        float mnew = m_run;
#pragma unroll
        for (int w2 = 0; w2 < NW; ++w2) mnew = fmaxf(mnew, red[w2]);
        const float alpha = expf(m_run - mnew);  // exp(-inf) = 0 on the first chunk
        m_run = mnew;
        l_loc *= alpha;
        // ---- weights e * v_scale; running sum ----
        if constexpr (S::kLaneSums) {
            if (own < n) {
                const float e = expf(own_sc - mnew);
                l_loc = l_loc + e;
                wsh[own] = e * own_vs;
            }
        } else {
            for (int pl = t; pl < n; pl += kThreads) {
                const int slot = slot_of(c * CH + pl);
                const float e = expf(wsh[pl] - mnew);
                l_loc = l_loc + e;
                wsh[pl] = e * vsb[slot];
            }
        }
        __syncthreads();
        // ---- values ----
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[e] *= alpha;
#pragma unroll
        for (int p = 0; p < S::VP; ++p) {
            const int pl = p * S::VPP + vpos;
            if (pl < n) {
                const float wgt = wsh[pl];
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[e] += wgt * i8_at(vr[p][e >> 2], e & 3);
            }
        }
        if (c + 1 < c_end) load_v(c + 1);  // lands during the next scores
        __syncthreads();
    }

    // ---- reduce over the lanes sharing a V column slice ----
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = ndl::wave_sum_from<S::VL>(acc[e]);
    if (lane < S::VL) {
#pragma unroll
        for (int e = 0; e < 16; ++e) vred[wave][lane * 16 + e] = acc[e];
    }
    const float wl = wave_sum(l_loc);
    if (lane == 0) red[wave] = wl;
    __syncthreads();
    for (int col = t; col < VD; col += kThreads) {
        float s = 0.0f, l = 0.0f;
#pragma unroll
        for (int w2 = 0; w2 < NW; ++w2) {
            s += vred[w2][col];
            l += red[w2];
        }
        if (splits == 1) {
            out[qi * size_t(g.H) * VD + size_t(kvh) * VD + col] = bad ? NAN : s / l;
        } else {
            part_o[((qi * g.H + kvh) * size_t(splits) + split) * VD + col] = s;
            if (col == 0) {
                float *ml = part_ml + ((qi * g.H + kvh) * size_t(splits) + split) * 2;
                ml[0] = bad ? NAN : (c_begin < c_end ? m_run : -INFINITY);
                ml[1] = l;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Attention over the int8 cache on the matrix cores: grouped query heads
// (several queries per K/V row) and prompts (all rows over one block).
//
// A wave owns 16 NT query columns -- (row, head) pairs that share a kv head
// -- and walks chunks of 32 positions with its own online softmax; no barrier
// until the waves of a block, which take the chunks in turn, merge at the end.
//   scores  S[pos][col] = K Q^T: v_mfma 16x16, A = 16 positions' int8 rows, as
//           they lie in the cache, B = the wave's query columns.  With
//           quant_query the query is int8 codes times one scale a head, so
//           the dot is an exact integer (i32_16x16x64_i8, no conversion of
//           K at all); else the fp32 query is three bf16 pieces whose sum is
//           exactly the query (scaled by a power of two where it is so small
//           that they would be subnormal) and K's codes are exact in bf16.
//   values  O^T[v][col] = V^T P^T: a score tile's result layout (lane = column,
//           four positions a lane) is the B layout the product needs, so the
//           weights stay in their lanes, as three bf16 pieces whose sum is
//           exactly the fp32 weight; V's codes are exact in bf16.  MFMA c
//           takes V columns 4 n + c, so a lane's V bytes come as one dword a
//           position and no byte is moved between lanes.
// Every product is exact and the sums are fp32 (or int32): nothing is held in
// 16 bits.  (A bf16 piece has no bit below 2^-126: a column that has met V
// scales below 2^-64 only takes its softmax against a maximum 64 bits lower.)
// What bounds it is the VALU work of the softmax (about 22 operations a score)
// and V's conversion (1.5 a byte, shared by the wave's columns); the matrix
// cores need about a third of the time.
// Measured, MI355X, kernel traces with the merge launch where there is one,
// quant_query, against the per-position kernel that took these calls before (K
// and V converted to fp32 and multiplied in the VALU for each query head; a
// prompt's rows each walked their own span):
//   prompt, 12 on 2 heads, qk 48: 500 rows 52.7 -> 8.7 us, 1000 81 -> 13.2,
//   2000 236 -> 29.9, 3000 473 -> 55 (12 x 64 MHA: 50 / 128 / 389 / 802 -> 9.5
//   / 14.2 / 30.2 / 57)
//   decode, 12 on 2 heads: 64 sessions x 2048 32.8 -> 12.0 us (fp32 query 30.8
//   -> 13.2), 256 x 1024 45.3 -> 13.6, one session x 8192 24.9 -> 10.4; 8 on 4:
//   64 x 2048 27.9 -> 14.4; 16 on 2: 256 x 1024 86.8 -> 14.2
// Watching for small V scales costs 2 % of these and 0.1 us of the shortest (calls
// back to back: 64 sessions x 2048 11.6 -> 11.9 us, 2000 rows 26.3 -> 27.0, 3000 47.6
// -> 49.0).  Found out afterwards, by a second walk of the columns that need it,
// it costs half as much of long prompts, and 0.5 us of short spans in 16-wave blocks.
// Four waves a SIMD for one column tile: with 129 registers instead of 128, many
// short spans took up to a fifth longer (785 sessions of 31 positions, 8 on 4
// heads: 12.9 and 15.5 us).
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));
typedef int intx4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// High halves of two floats: (bf16 of a, bf16 of b) where both are exact.
__device__ inline uint32_t pack_hi(float a, float b)
{
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}

__device__ inline float trunc_hi(float a) { return __uint_as_float(__float_as_uint(a) & 0xffff0000u); }

// fmaxf of three (a NaN loses), without the copies the compiler makes of
// operands it cannot show to be quiet.
__device__ inline float max3(float a, float b, float c)
{
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// x0, x1 as three bf16 pairs that sum to them exactly (8 mantissa bits each).
__device__ inline void split3(float x0, float x1, uint32_t &h, uint32_t &m, uint32_t &l)
{
    h = pack_hi(x0, x1);
    const float r0 = x0 - trunc_hi(x0), r1 = x1 - trunc_hi(x1);
    m = pack_hi(r0, r1);
    l = pack_hi(r0 - trunc_hi(r0), r1 - trunc_hi(r1));
}

template <int QK, bool QQ, int NT, int NW, bool SHARED>
__global__ __launch_bounds__(NW * 64, NT == 1 ? 4 : 1) void attn_mm_kernel(
    Geom g, const uint8_t *__restrict__ kv, size_t kv_stride, const int32_t *__restrict__ lo_a,
    const int32_t *__restrict__ hi_a, const float *__restrict__ q, float scale2, int rows, int splits,
    float *__restrict__ out, float *__restrict__ part_o, float *__restrict__ part_ml)
{
    constexpr int VD = 64, SL = QK / 4;             // a lane's slice of a K row
    constexpr int KD = SL / 4;                      // its dwords (3 or 4)
    constexpr int COLS = SHARED ? 16 * NT : kMaxRep;  // merged columns
    constexpr int LD = VD + 4;
    static_assert(SHARED || NT == 1, "one query: at most kMaxRep columns");
    __shared__ __align__(16) float sc_s[NW][64];
    __shared__ __align__(16) float mo[NW][COLS][LD];
    __shared__ float mm[NW][COLS], ml[NW][COLS], mf[NW][COLS];

    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int n = lane & 15, qd = lane >> 4;
    const int R = g.H / g.KVH;
    const int kvh = blockIdx.x % g.KVH, split = blockIdx.x / g.KVH;
    // later tiles of a prompt have the longer spans: they start first
    const int tile = SHARED ? int(gridDim.y) - 1 - int(blockIdx.y) : int(blockIdx.y);
    const uint8_t *blk = SHARED ? kv : kv + size_t(tile) * kv_stride;
    const int8_t *kb = reinterpret_cast<const int8_t *>(blk) + size_t(kvh) * g.cap * QK;
    const int8_t *vb = reinterpret_cast<const int8_t *>(blk + g.v_off) + size_t(kvh) * g.cap * VD;
    const float *ksb = reinterpret_cast<const float *>(blk + g.ks_off) + size_t(kvh) * g.cap;
    const float *vsb = reinterpret_cast<const float *>(blk + g.vs_off) + size_t(kvh) * g.cap;
    const uint32_t cap = uint32_t(g.cap);

    // ---- the wave's columns: their spans and query operands ----
    const int ncols = SHARED ? rows * R : R;  // columns of this kv head (and query)
    // f / R of a column f < 2^20: (f + 1/2) / R is 1/16 or more away from an
    // integer (R <= 8), and its float error is below 2^20 2^-22 / R
    const float inv_r = 1.0f / float(R);
    auto row_of = [&](int f) { return SHARED ? int((float(f) + 0.5f) * inv_r) : tile; };
    uint32_t lo[NT], hi[NT];
    bool bad[NT];
    float cf[NT];                              // column factor of a score, in bits
    intx4_t qi[NT];                            // QQ: codes
    uint32_t qp[NT][3][KD == 3 ? 6 : 8];       // else: bf16 pieces
    uint32_t ulo = 0xffffffffu, uhi = 0;
    float spans = 0.0f;
#pragma unroll
    for (int x = 0; x < NT; ++x) {
        const int f0 = (SHARED ? tile * (16 * NT) + 16 * x : 0) + n;
        const int f = f0 < ncols ? f0 : ncols - 1;  // past the end: a copy, not written
        const int row = row_of(f);
        const int head = kvh * R + (SHARED ? f - row * R : f);
        const int l0 = lo_a[row], h0 = hi_a[row];
        // h0 - l0 cannot overflow where l0 >= 0 and h0 >= l0
        bad[x] = l0 < 0 || h0 < l0 || h0 - l0 >= g.cap;
        lo[x] = bad[x] ? 0xffffffffu : uint32_t(l0);
        hi[x] = bad[x] ? 0u : uint32_t(h0);
        if (!bad[x]) {
            ulo = min(ulo, lo[x]);
            uhi = max(uhi, hi[x]);
            spans += float(h0 - l0 + 1);
        }
        const float *qh = q + (size_t(row) * g.H + head) * QK + qd * SL;
        float v[SL];
#pragma unroll
        for (int e = 0; e < SL; ++e) v[e] = qh[e];
        if constexpr (QQ) {
            // quant_rows (model.rs:289-293): the codes and the head's scale
            float a = 0.0f;
#pragma unroll
            for (int e = 0; e < SL; e += 2) a = max3(a, __builtin_fabsf(v[e]), __builtin_fabsf(v[e + 1]));
            a = fmaxf(a, ndl::wave_xor<16>(a));
            a = fmaxf(a, ndl::wave_xor<32>(a));
            const float qs = a > 0.0f ? a / 127.0f : 1.0f;
            const float inv = 1.0f / qs;
            float nan = 0.0f;  // NaN where a code is (an infinite y, of a subnormal scale, has one)
            uint32_t dw[4] = {0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < SL; ++e) {
                // quant_code: half away from zero is truncation after adding
                // the float below a half, for every |y| < 2^22
                const float y = v[e] * inv;
                const float r = __builtin_amdgcn_fmed3f(y + copysignf(0.49999997f, y), -128.0f, 127.5f);
                nan = y != y ? y : nan;
                dw[e >> 2] |= (uint32_t(int32_t(r)) & 0xffu) << (8 * (e & 3));
            }
            nan += ndl::wave_xor<16>(nan);
            nan += ndl::wave_xor<32>(nan);
            qi[x] = intx4_t{int(dw[0]), int(dw[1]), int(dw[2]), int(dw[3])};
            cf[x] = qs * scale2 + nan;
        } else {
            // a bf16 piece has no bit below 2^-126: a head of small values goes
            // in 2^100 times as large
            cf[x] = scale2;
            float a = 0.0f;
#pragma unroll
            for (int e = 0; e < SL; ++e) a += __builtin_fabsf(v[e]);
            if (__any(a < 0x1p-100f)) {
                a += ndl::wave_xor<16>(a);
                a += ndl::wave_xor<32>(a);
                const bool small = a < 0x1p-100f;
                if (small) cf[x] = scale2 * 0x1p-100f;
#pragma unroll
                for (int e = 0; e < SL; ++e) v[e] *= small ? 0x1p100f : 1.0f;
            }
#pragma unroll
            for (int e = 0; e < SL; e += 2) split3(v[e], v[e + 1], qp[x][0][e / 2], qp[x][1][e / 2], qp[x][2][e / 2]);
        }
    }
    // the union of the columns' spans (the same in all four lane quarters)
    {
        auto umin = [&](uint32_t &a, uint32_t b) { a = min(a, b); };
        auto umax = [&](uint32_t &a, uint32_t b) { a = max(a, b); };
        umin(ulo, uint32_t(ndl::wave_xor_int<1>(int(ulo)))), umax(uhi, uint32_t(ndl::wave_xor_int<1>(int(uhi))));
        umin(ulo, uint32_t(ndl::wave_xor_int<2>(int(ulo)))), umax(uhi, uint32_t(ndl::wave_xor_int<2>(int(uhi))));
        umin(ulo, uint32_t(ndl::wave_xor_int<4>(int(ulo)))), umax(uhi, uint32_t(ndl::wave_xor_int<4>(int(uhi))));
        umin(ulo, uint32_t(ndl::wave_xor_int<8>(int(ulo)))), umax(uhi, uint32_t(ndl::wave_xor_int<8>(int(uhi))));
        spans = ndl::group_sum<16>(spans);
        ulo = __builtin_amdgcn_readfirstlane(ulo);
        uhi = __builtin_amdgcn_readfirstlane(uhi);
        spans = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(spans)));
    }
    const bool any = uhi >= ulo;
    // Rows of a prompt overlap, and the wave walks the union of their spans.
    // Rows that share little (a caller's own lo and hi) would make the union
    // longer than the rows together: then each chunk starts where some row
    // still has a position, so no more chunks are walked than the rows have.
    const bool sparse = SHARED && any && float(uhi - ulo) + 1.0f > spans / float(R) + 64.0f;
    const uint32_t step = uint32_t(splits) * NW;  // waves that share the walk
    uint32_t p0 = ulo, s0 = 0;
    bool more = any;
    const uint32_t step_mod = (32u * step) % cap;
    auto next_start = [&](uint32_t from) {  // first position >= from of any column
        uint32_t c = 0xffffffffu;
#pragma unroll
        for (int x = 0; x < NT; ++x)
            if (!bad[x] && hi[x] >= from) c = min(c, max(lo[x], from));
        c = min(c, uint32_t(ndl::wave_xor_int<1>(int(c))));
        c = min(c, uint32_t(ndl::wave_xor_int<2>(int(c))));
        c = min(c, uint32_t(ndl::wave_xor_int<4>(int(c))));
        c = min(c, uint32_t(ndl::wave_xor_int<8>(int(c))));
        return uint32_t(__builtin_amdgcn_readfirstlane(c));
    };
    auto advance = [&](uint32_t k, uint32_t mod) {  // k chunks on
        if (!sparse) {
            // p0 - ulo < 2^31 and 32 k < 2^31: no wrap
            p0 += 32u * k;
            s0 += mod;
            if (s0 >= cap) s0 -= cap;
            more = p0 <= uhi && p0 >= ulo;
        } else {
            for (uint32_t i = 0; i < k && more; ++i) {
                p0 = next_start(p0 + 32u);  // positions end below 2^31
                more = p0 != 0xffffffffu;
            }
            if (more) s0 = p0 % cap;
        }
    };
    if (any) {
        s0 = ulo % cap;
        const uint32_t first = uint32_t(split) * NW + uint32_t(w);
        if (first) advance(first, (32u * first) % cap);
    }

    uint32_t kr[2][KD], vr[8];
    float scr = 0.0f;
    // a chunk inside the ring: scalar base, lane and pass offsets; across its
    // end (or in a ring below a chunk): each position's slot
    auto slot_of = [&](uint32_t off) { return (s0 + off) % cap; };
    auto load_k = [&]() {
        if (s0 + 32u <= cap) {
            const int8_t *p = kb + size_t(s0) * QK;
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int d = 0; d < KD; ++d)
                    kr[a][d] = *reinterpret_cast<const uint32_t *>(p + (n * QK + qd * SL) + (16 * a * QK + 4 * d));
            scr = *(lane < 32 ? ksb + s0 + lane : vsb + s0 + (lane - 32));
        } else {
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                const int8_t *p = kb + size_t(slot_of(16 * a + n)) * QK + qd * SL;
#pragma unroll
                for (int d = 0; d < KD; ++d) kr[a][d] = *reinterpret_cast<const uint32_t *>(p + 4 * d);
            }
            scr = (lane < 32 ? ksb : vsb)[slot_of(lane & 31)];
        }
    };
    auto load_v = [&]() {
        if (s0 + 32u <= cap) {
            const int8_t *p = vb + size_t(s0) * VD;
#pragma unroll
            for (int j = 0; j < 8; ++j)
                vr[j] = *reinterpret_cast<const uint32_t *>(p + (4 * qd * VD + 4 * n) + (16 * (j >> 2) + (j & 3)) * VD);
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                vr[j] = *reinterpret_cast<const uint32_t *>(
                    vb + size_t(slot_of(16 * (j >> 2) + 4 * qd + (j & 3))) * VD + 4 * n);
        }
    };
    // loads are never conditional: past the last chunk they reread a slot
    load_k();
    load_v();

    float m_run[NT], l_run[NT];
    floatx4_t acc[NT][4];
#pragma unroll
    for (int x = 0; x < NT; ++x) {
        m_run[x] = -INFINITY;
        l_run[x] = 0.0f;
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[x][c] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }
    // As long as every V scale of the column is below 2^-64 its sums are taken
    // against a maximum 64 bits lower: its weights' pieces are normal numbers.
    bool low[NT], any_low = true;
#pragma unroll
    for (int x = 0; x < NT; ++x) low[x] = true;

    while (more) {
        const uint32_t pc = p0;
        // positions of the chunk whose V scale is 2^-64 or more
        const uint32_t normal = uint32_t(__ballot(!(__builtin_fabsf(scr) < 0x1p-64f)) >> 32);
        // the chunk's scales, from position order to the score tiles' rows
        sc_s[w][lane] = scr;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        floatx4_t ks[2], vs[2];
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            ks[a] = *reinterpret_cast<const floatx4_t *>(&sc_s[w][16 * a + 4 * qd]);
            vs[a] = *reinterpret_cast<const floatx4_t *>(&sc_s[w][32 + 16 * a + 4 * qd]);
        }
        __builtin_amdgcn_wave_barrier();
        // ---- scores ----
        float s[NT][8];
        if constexpr (QQ) {
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                // query scale before K scale: a dot times a large K scale would
                // overflow where the reference's order, query codes scaled, does not
                const intx4_t kf{int(kr[a][0]), int(kr[a][1]), int(kr[a][2]), KD == 3 ? 0 : int(kr[a][KD - 1])};
#pragma unroll
                for (int x = 0; x < NT; ++x) {
                    const intx4_t d = __builtin_amdgcn_mfma_i32_16x16x64_i8(kf, qi[x], intx4_t{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; ++i) s[x][4 * a + i] = (float(d[i]) * cf[x]) * ks[a][i];
                }
            }
        } else {
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                uint32_t kp[2 * KD];
#pragma unroll
                for (int d = 0; d < KD; ++d) {
                    kp[2 * d] = pack_hi(i8_at(kr[a][d], 0), i8_at(kr[a][d], 1));
                    kp[2 * d + 1] = pack_hi(i8_at(kr[a][d], 2), i8_at(kr[a][d], 3));
                }
                const bf16x8_t k0 = __builtin_bit_cast(bf16x8_t, u32x4_t{kp[0], kp[1], kp[2], kp[3]});
#pragma unroll
                for (int x = 0; x < NT; ++x) {
                    floatx4_t d{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int pc3 = 2; pc3 >= 0; --pc3) {  // the small pieces first
                        const uint32_t *qq = qp[x][pc3];
                        // qk 48: a lane's last four codes, doubled to the 32-wide
                        // product's eight against four zeros of the query
                        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(bf16x8_t, u32x4_t{kp[4], kp[5], kp[2 * KD - 2], kp[2 * KD - 1]}),
                            __builtin_bit_cast(bf16x8_t, KD == 3 ? u32x4_t{qq[4], qq[5], 0u, 0u}
                                                                 : u32x4_t{qq[4], qq[5], qq[2 * KD - 2], qq[2 * KD - 1]}),
                            d, 0, 0, 0);
                        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            k0, __builtin_bit_cast(bf16x8_t, u32x4_t{qq[0], qq[1], qq[2], qq[3]}), d, 0, 0, 0);
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) s[x][4 * a + i] = (d[i] * cf[x]) * ks[a][i];
                }
            }
        }
        advance(step, step_mod);
        load_k();  // lands during the softmax and the values
        // ---- softmax: each lane its column's eight positions ----
        bool inside = true;
#pragma unroll
        for (int x = 0; x < NT; ++x) inside = inside && !bad[x] && lo[x] <= pc && hi[x] >= pc + 31u;
        const bool full = __all(inside);
        if (!full) {
#pragma unroll
            for (int x = 0; x < NT; ++x)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const uint32_t p = pc + uint32_t(16 * (j >> 2) + 4 * qd + (j & 3));
                    if (p < lo[x] || p > hi[x]) s[x][j] = -INFINITY;
                }
        }
        bool grew = false;
        float m_new[NT];
#pragma unroll
        for (int x = 0; x < NT; ++x) {
            const float m8 = max3(max3(s[x][0], s[x][1], s[x][2]), max3(s[x][3], s[x][4], s[x][5]),
                                  max3(s[x][6], s[x][7], m_run[x]));
            // over the four lane quarters: each swap returns the pair
            const auto s16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(m8), __float_as_uint(m8), false, false);
            const float m16 = max3(__uint_as_float(s16[0]), __uint_as_float(s16[1]), m8);
            const auto s32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(m16), __float_as_uint(m16), false, false);
            m_new[x] = max3(__uint_as_float(s32[0]), __uint_as_float(s32[1]), m16);
            grew = grew || m_new[x] > m_run[x];
        }
        bool up[NT];
#pragma unroll
        for (int x = 0; x < NT; ++x) up[x] = false;
        if (any_low) {
            bool still = false;
#pragma unroll
            for (int x = 0; x < NT; ++x) {
                // the column's own of them, from its first position to its last (one
                // span for all columns of a row: scalar)
                const uint32_t first = max(SHARED ? lo[x] : ulo, pc), last = min(SHARED ? hi[x] : uhi, pc + 31u);
                const uint32_t own = (normal >> ((first - pc) & 31u)) << ((first - last - 1u) & 31u);
                up[x] = low[x] && ((SHARED && bad[x]) || (first <= last && own != 0));
                low[x] = low[x] && !up[x];
                grew = grew || up[x];
                still = still || low[x];
            }
            any_low = __any(still);
        }
        if (__any(grew)) {
#pragma unroll
            for (int x = 0; x < NT; ++x) {
                float al = m_new[x] > m_run[x] ? __builtin_amdgcn_exp2f(m_run[x] - m_new[x]) : 1.0f;
                al = up[x] ? al * 0x1p-64f : al;
                m_run[x] = m_new[x];
                l_run[x] *= al;
#pragma unroll
                for (int c = 0; c < 4; ++c) acc[x][c] *= al;
            }
        }
        uint32_t pp[NT][3][4];
#pragma unroll
        for (int x = 0; x < NT; ++x) {
            const float mu = (m_run[x] == -INFINITY ? 0.0f : m_run[x]) - (low[x] ? 64.0f : 0.0f);
            float wt[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float e = __builtin_amdgcn_exp2f(s[x][j] - mu);
                l_run[x] += e;
                wt[j] = e * vs[j >> 2][j & 3];
            }
            if (!full) {
                // a slot no row reads may hold anything, a NaN scale too
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const uint32_t p = pc + uint32_t(16 * (j >> 2) + 4 * qd + (j & 3));
                    if (p < lo[x] || p > hi[x]) wt[j] = 0.0f;
                }
            }
#pragma unroll
            for (int j = 0; j < 8; j += 2)
                split3(wt[j], wt[j + 1], pp[x][0][j / 2], pp[x][1][j / 2], pp[x][2][j / 2]);
        }
        // ---- values ----
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            uint32_t vp[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) vp[j] = pack_hi(i8_at(vr[2 * j], c), i8_at(vr[2 * j + 1], c));
            const bf16x8_t vf = __builtin_bit_cast(bf16x8_t, u32x4_t{vp[0], vp[1], vp[2], vp[3]});
#pragma unroll
            for (int x = 0; x < NT; ++x)
#pragma unroll
                for (int pc3 = 2; pc3 >= 0; --pc3)
                    acc[x][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        vf, __builtin_bit_cast(bf16x8_t, u32x4_t{pp[x][pc3][0], pp[x][pc3][1], pp[x][pc3][2], pp[x][pc3][3]}),
                        acc[x][c], 0, 0, 0);
        }
        load_v();  // lands during the next scores
    }

    // ---- merge the block's waves ----
#pragma unroll
    for (int x = 0; x < NT; ++x) {
        float l = l_run[x];
        l += ndl::wave_xor<16>(l);
        l += ndl::wave_xor<32>(l);
        const int col = 16 * x + n;
        if (col < COLS) {
            if (qd == 0) {
                mm[w][col] = bad[x] ? NAN : m_run[x] - (low[x] ? 64.0f : 0.0f);
                ml[w][col] = l;
            }
            // lane (n, qd) holds V columns 16 qd + 4 i + c
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<floatx4_t *>(&mo[w][col][16 * qd + 4 * i]) =
                    floatx4_t{acc[x][0][i], acc[x][1][i], acc[x][2][i], acc[x][3][i]};
        }
    }
    __syncthreads();
    for (int o = t; o < NW * COLS; o += NW * 64) {
        const int i = o / COLS, col = o % COLS;
        float M = -INFINITY;
#pragma unroll
        for (int j = 0; j < NW; ++j) M = fmaxf(M, mm[j][col]);
        const float m = mm[i][col];
        // -inf: the wave's sums are 0, or NaN where a score was; NaN: a bad span
        mf[i][col] = m == -INFINITY ? 1.0f : exp2f(m - M);
    }
    __syncthreads();
    for (int col = w; col < COLS; col += NW) {  // a wave a column, a lane a value
        const int f = (SHARED ? tile * (16 * NT) : 0) + col;
        if (f >= ncols) break;
        const int row = __builtin_amdgcn_readfirstlane(row_of(f));
        const int head = kvh * R + (SHARED ? f - row * R : f);
        float O = 0.0f, L = 0.0f;
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            O += mo[i][col][lane] * mf[i][col];
            L += ml[i][col] * mf[i][col];
        }
        const size_t oh = size_t(row) * g.H + head;
        if (splits == 1) {
            out[oh * VD + lane] = O / L;
        } else {
            part_o[(oh * splits + split) * VD + lane] = O;
            if (lane == 0) {
                float M = -INFINITY;
                for (int i = 0; i < NW; ++i) M = fmaxf(M, mm[i][col]);
                float *p = part_ml + (oh * splits + split) * 2;
                p[0] = L != L ? NAN : M;
                p[1] = L;
            }
        }
    }
}

// Merge chunk partials: out = sum_c o_c e^(m_c - M) / sum_c l_c e^(m_c - M);
// with BASE2, powers of two (the matrix-core kernel's maxima are in bits).
template <bool BASE2>
__global__ __launch_bounds__(64) void attn_combine_kernel(Geom g, int nchunks,
                                                               const float *__restrict__ part_o,
                                                               const float *__restrict__ part_ml,
                                                               float *__restrict__ out)
{
    // a lane a column (v is 64 wherever attention is split); the partials'
    // factors 64 at a time in the lanes, four partials loaded ahead
    const size_t qi = blockIdx.y;
    const int head = blockIdx.x, lane = threadIdx.x;
    const size_t base = (qi * g.H + head) * size_t(nchunks);
    const float *po = part_o + base * 64 + lane;
    const float2 *mls = reinterpret_cast<const float2 *>(part_ml) + base;
    auto load_ml = [&](int c) { return c < nchunks ? mls[c] : make_float2(-INFINITY, 0.0f); };
    float2 ml = load_ml(lane);
    float o[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) o[u] = po[size_t(min(u, nchunks - 1)) * 64];
    float M = ml.x;
    for (int c = lane + 64; c < nchunks; c += 64) M = fmaxf(M, mls[c].x);
    M = wave_max(M);
    float O = 0.0f, L = 0.0f;
    for (int c0 = 0; c0 < nchunks; c0 += 64) {
        if (c0) ml = load_ml(c0 + lane);
        const float f = ml.x == -INFINITY ? 0.0f : (BASE2 ? exp2f(ml.x - M) : expf(ml.x - M));
        const float l = ml.x == -INFINITY ? 0.0f : ml.y;
        const int nc = min(64, nchunks - c0);
        for (int c = 0; c < nc; c += 4) {
            float next[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) next[u] = po[size_t(min(c0 + c + 4 + u, nchunks - 1)) * 64];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                // past the end: lane 63's or -inf's factor, left out
                const float fc = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(f), min(c + u, 63)));
                const float lc = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(l), min(c + u, 63)));
                if (c + u < nc) {
                    O += o[u] * fc;
                    L += lc * fc;
                }
                o[u] = next[u];
            }
        }
    }
    out[(qi * size_t(g.H) + head) * 64 + lane] = O / L;
}

using AttnFn = void (*)(dim3, hipStream_t, Geom, const uint8_t *, size_t, const int32_t *,
                        const int32_t *, const float *, float, int, int, int, float *, float *, float *);

template <int QK>
void launch_attn(dim3 grid, hipStream_t s, Geom g, const uint8_t *kv, size_t stride,
                 const int32_t *lo, const int32_t *hi, const float *q, float scale, int qq,
                 int, int splits, float *out, float *po, float *pml)
{
    hipLaunchKernelGGL((attn_i8_kernel<QK, 64>), grid, dim3(kThreads), 0, s, g, kv, stride, lo, hi, q,
                       scale, qq, splits, out, po, pml);
}

template <int QK, int NT, int NW, bool SHARED>
void launch_mm(dim3 grid, hipStream_t s, Geom g, const uint8_t *kv, size_t stride, const int32_t *lo,
               const int32_t *hi, const float *q, float scale, int qq, int rows, int splits, float *out,
               float *po, float *pml)
{
    const float scale2 = float(double(scale) * 1.4426950408889634);  // scores in bits: e^s = 2^(s log2 e)
    if (qq)
        hipLaunchKernelGGL((attn_mm_kernel<QK, true, NT, NW, SHARED>), grid, dim3(NW * 64), 0, s, g, kv,
                           stride, lo, hi, q, scale2, rows, splits, out, po, pml);
    else
        hipLaunchKernelGGL((attn_mm_kernel<QK, false, NT, NW, SHARED>), grid, dim3(NW * 64), 0, s, g, kv,
                           stride, lo, hi, q, scale2, rows, splits, out, po, pml);
}

// Instantiated: qk 48 (the shipped v3 geometry) and 64 (the MHA cache), v 64,
// query heads per kv head 1, 2, 3, 4, 6, 8.
bool attn_shape(int rep, int qk, int vd)
{
    const bool r = rep == 1 || rep == 2 || rep == 3 || rep == 4 || rep == 6 || rep == 8;
    return r && (qk == 48 || qk == 64) && vd == 64;
}

// The matrix-core kernel takes every prompt but the shortest of one query head a
// kv head (figures at the rule), and every decode call with two or more query
// heads a kv head (figures at the kernel).  One query head a kv
// head stays with attn_i8_kernel: its column tile would be 1/16 full, and
// where the caches stream from HBM it is the faster of the two (12 x 64, 256
// sessions x 1024: 70 against 77-85 us; 64 x 512: 11.5 against 11.6-13.1).
constexpr int kMmMinRep = 2;

}  // namespace

extern "C" {

size_t nd_kv_v_offset(const nd_kv_geom *g)
{
    return nd::align_up(size_t(g->num_kv_heads) * g->cap * g->qk_head_dim, 256);
}

size_t nd_kv_ks_offset(const nd_kv_geom *g)
{
    return nd_kv_v_offset(g) + nd::align_up(size_t(g->num_kv_heads) * g->cap * g->v_head_dim, 256);
}

size_t nd_kv_vs_offset(const nd_kv_geom *g)
{
    return nd_kv_ks_offset(g) + nd::align_up(size_t(g->num_kv_heads) * g->cap * 4, 256);
}

size_t nd_kv_block_bytes(const nd_kv_geom *g)
{
    return nd_kv_vs_offset(g) + nd::align_up(size_t(g->num_kv_heads) * g->cap * 4, 256);
}

size_t nd_kv_f32_v_offset(const nd_kv_geom *g)
{
    return nd::align_up(size_t(g->num_kv_heads) * g->cap * g->qk_head_dim * 4, 256);
}

size_t nd_kv_f32_block_bytes(const nd_kv_geom *g)
{
    return nd_kv_f32_v_offset(g) + nd::align_up(size_t(g->num_kv_heads) * g->cap * g->v_head_dim * 4, 256);
}

int nd_kv_write_f32(nd_ctx *ctx, const nd_kv_geom *g, void *kv, size_t kv_stride, size_t count,
                    const int32_t *pos, const float *k, const float *v)
{
    ND_ENTER(ctx);
    if (int rc = check_geom(g)) return rc;
    if (count == 0) return ND_OK;
    ND_REQUIRE(kv && pos && k && v, "null buffer");
    ND_REQUIRE(count <= 0x7fffffff, "count too large");
    Geom kg = make_geom(g);
    kg.v_off = nd_kv_f32_v_offset(g);
    dim3 grid(unsigned(count), unsigned(g->num_kv_heads));
    hipLaunchKernelGGL(kv_write_f32_kernel, grid, dim3(64), 0, ctx->stream, kg,
                       static_cast<uint8_t *>(kv), kv_stride, pos, k, v);
    return nd::check_launch("kv_write_f32");
}

int nd_fake_quant(nd_ctx *ctx, float *x, size_t rows, size_t dim)
{
    ND_ENTER(ctx);
    if (rows == 0) return ND_OK;
    ND_REQUIRE(x && dim > 0 && dim <= (1u << 20), "bad arguments");
    const size_t blocks = (rows + 3) / 4;
    ND_REQUIRE(blocks <= 0x7fffffff, "too many rows");
    hipLaunchKernelGGL(fake_quant_kernel, dim3(unsigned(blocks)), dim3(kThreads), 0, ctx->stream, x,
                       rows, int(dim));
    return nd::check_launch("fake_quant");
}

int nd_quantize_rows(nd_ctx *ctx, const float *x, size_t rows, size_t head_dim, int8_t *ints,
                     float *scales)
{
    ND_ENTER(ctx);
    if (rows == 0) return ND_OK;
    ND_REQUIRE(x && ints && scales && head_dim > 0 && head_dim <= (1u << 20), "bad arguments");
    const size_t blocks = (rows + 3) / 4;
    ND_REQUIRE(blocks <= 0x7fffffff, "too many rows");
    hipLaunchKernelGGL(quantize_rows_kernel, dim3(unsigned(blocks)), dim3(kThreads), 0, ctx->stream,
                       x, rows, int(head_dim), ints, scales);
    return nd::check_launch("quantize_rows");
}

int nd_kv_write(nd_ctx *ctx, const nd_kv_geom *g, void *kv, size_t kv_stride, size_t count,
                const int32_t *pos, const float *k, const float *v)
{
    ND_ENTER(ctx);
    if (int rc = check_geom(g)) return rc;
    if (count == 0) return ND_OK;
    ND_REQUIRE(kv && pos && k && v, "null buffer");
    ND_REQUIRE(count <= 0x7fffffff, "count too large");
    dim3 grid(unsigned(count), unsigned(g->num_kv_heads));
    hipLaunchKernelGGL(kv_write_kernel, grid, dim3(128), 0, ctx->stream, make_geom(g),
                       static_cast<uint8_t *>(kv), kv_stride, pos, k, v);
    return nd::check_launch("kv_write");
}

}  // extern "C"

namespace {

// nd_attend_step_i8 with its split-K partials either in the context's
// growable workspace (fixed == nullptr) or in `fixed`, `fixed_floats` long.
int attend_i8(nd_ctx *ctx, const nd_kv_geom *g, const void *kv, size_t kv_stride, size_t count,
              const int32_t *lo, const int32_t *hi, const float *q, float scale, int quant_query,
              float *out, float *fixed, size_t fixed_floats)
{
    ND_ENTER(ctx);
    if (int rc = check_geom(g)) return rc;
    if (count == 0) return ND_OK;
    ND_REQUIRE(kv && lo && hi && q && out, "null buffer");
    ND_REQUIRE(count <= 65535, "count %zu above 65535", count);
    ND_REQUIRE((reinterpret_cast<uintptr_t>(kv) & 255) == 0 && kv_stride % 256 == 0,
               "kv blocks must be 256-byte aligned");
    const int rep = g->num_heads / g->num_kv_heads;
    ND_REQUIRE(attn_shape(rep, g->qk_head_dim, g->v_head_dim),
               "no attention kernel for repeat %d, qk %d, v %d", rep, g->qk_head_dim, g->v_head_dim);
    // Split each span across blocks only when (query, kv head) pairs cannot
    // give every CU a few blocks; the split partials merge in a second pass.
    const size_t pairs = count * size_t(g->num_kv_heads);
    const size_t cus = size_t(ctx->num_cus > 0 ? ctx->num_cus : 256);
    const size_t want = cus * 4;
    // a split covers at least 512 positions (256 with more than two query
    // heads a kv head): with one query head, splits of one 256-position
    // chunk measured slower at one session (ctx 512: 13.1 against 10.6 us,
    // ctx 8192: 20.4 against 14.9), the merge costing more than they save
    const size_t span_min = rep <= 2 ? 512 : 256;
    const size_t max_splits = (size_t(g->cap) + span_min - 1) / span_min;
    size_t splits = pairs >= want ? 1 : (want + pairs - 1) / pairs;
    if (splits > max_splits) splits = max_splits;
    if (splits > 65535) splits = 65535;
    if (fixed && splits > 1) {
        const size_t need = count * size_t(g->num_heads) * splits * (g->v_head_dim + 2);
        ND_REQUIRE(need <= fixed_floats,
                   "split-K partials need %zu floats (%zu queries x %d heads x %zu splits x "
                   "(%d + 2)); the no-allocation scratch holds %zu",
                   need, count, g->num_heads, splits, g->v_head_dim, fixed_floats);
    }
    const bool q48 = g->qk_head_dim == 48;
    bool base2 = true;
    AttnFn fn;
    dim3 grid;
    // A short prompt with one query head a kv head, in blocks of one row: as long
    // as each has a CU of its own, a tile of 16 rows only waits longer (us, 12
    // heads, matrix cores / rows: 8 rows 5.0 / 4.3, 20 rows 5.5 / 4.4, 17 rows in a
    // ring of 243 4.9 / 4.5, 10 in one of 776 7.8 / 7.0; 26 rows 5.4 / 5.5, 46 rows
    // 5.2 / 6.3, 16 in a ring of 1995 7.4 / 8.4, 12 in one of 3445 7.4 / 9.1)
    const bool few_rows = rep < kMmMinRep && pairs * max_splits <= cus;
    if (kv_stride == 0 && count > 1 && !few_rows) {
        // A prompt's rows over one block.  Two column tiles a wave share V's
        // conversion once that leaves four blocks a CU (3000 rows, 12 on 2:
        // 53 against 57 us; 2000: 31 against 29); with fewer than two
        // single-tile blocks a CU, eight waves a block (500 rows: 9.3 against
        // 14.3 us with four; 1000: 14.7 against 12.8)
        const size_t cols = count * size_t(rep);
        const size_t kvh = size_t(g->num_kv_heads);
        const bool wide = (cols + 31) / 32 * kvh >= 4 * cus;
        const size_t tiles = wide ? (cols + 31) / 32 : (cols + 15) / 16;
        const size_t nw = !wide && tiles * kvh < 2 * cus ? 8 : 4;
        const size_t fill = (cus * 8 + tiles * g->num_kv_heads * nw - 1) / (tiles * g->num_kv_heads * nw);
        if (splits > fill) splits = fill;
        grid = dim3(unsigned(g->num_kv_heads * splits), unsigned(tiles));
        fn = wide      ? (q48 ? launch_mm<48, 2, 4, true> : launch_mm<64, 2, 4, true>)
             : nw == 4 ? (q48 ? launch_mm<48, 1, 4, true> : launch_mm<64, 1, 4, true>)
                       : (q48 ? launch_mm<48, 1, 8, true> : launch_mm<64, 1, 8, true>);
    } else if (rep >= kMmMinRep) {
        // Two waves a SIMD or more, from one block where it can be: 16-wave
        // blocks below 8 waves a CU (64 sessions x 2 heads x 512: 7.4 against
        // 9.7 us with four waves and a merge launch), 4-wave blocks above
        // (256 x 2 x 1024: 15.3 against 17.3); no split leaves a wave without
        // a chunk, and a ring of up to four chunks has none for more waves
        // (172 x 2 heads x 8 positions: 10.5 us with 16 waves, 5.8 so)
        const bool deep = pairs * 4 < cus * 8 && g->cap > 128;
        const size_t nw = deep ? 16 : 4;
        const size_t fill = (cus * 8 + pairs * nw - 1) / (pairs * nw);
        const size_t most = (size_t(g->cap) + 32 * nw - 1) / (32 * nw);
        if (splits > fill) splits = fill;
        if (splits > most) splits = most;
        grid = dim3(unsigned(g->num_kv_heads * splits), unsigned(count));
        fn = deep ? (q48 ? launch_mm<48, 1, 16, false> : launch_mm<64, 1, 16, false>)
                  : (q48 ? launch_mm<48, 1, 4, false> : launch_mm<64, 1, 4, false>);
    } else {
        grid = dim3(unsigned(splits), unsigned(g->num_kv_heads), unsigned(count));
        base2 = false;
        fn = q48 ? launch_attn<48> : launch_attn<64>;
    }
    float *po = nullptr, *pml = nullptr;
    if (splits > 1) {
        void *wsp = nullptr;
        const size_t n_o = count * size_t(g->num_heads) * splits * g->v_head_dim;
        const size_t n_ml = count * size_t(g->num_heads) * splits * 2;
        if (fixed) {
            wsp = fixed;
        } else if (int rc = nd::workspace(ctx, (n_o + n_ml) * sizeof(float), &wsp)) {
            return rc;
        }
        po = static_cast<float *>(wsp);
        pml = po + n_o;
    }
    fn(grid, ctx->stream, make_geom(g), static_cast<const uint8_t *>(kv), kv_stride, lo, hi, q,
       scale, quant_query, int(count), int(splits), out, po, pml);
    if (int rc = nd::check_launch("attn_i8")) return rc;
    if (splits > 1) {
        const dim3 cg(unsigned(g->num_heads), unsigned(count));
        if (base2)
            hipLaunchKernelGGL(attn_combine_kernel<true>, cg, dim3(64), 0, ctx->stream, make_geom(g),
                               int(splits), po, pml, out);
        else
            hipLaunchKernelGGL(attn_combine_kernel<false>, cg, dim3(64), 0, ctx->stream, make_geom(g),
                               int(splits), po, pml, out);
        return nd::check_launch("attn_combine");
    }
    return ND_OK;
}

}  // namespace

extern "C" {

int nd_attend_step_i8(nd_ctx *ctx, const nd_kv_geom *g, const void *kv, size_t kv_stride,
                      size_t count, const int32_t *lo, const int32_t *hi, const float *q,
                      float scale, int quant_query, float *out)
{
    return attend_i8(ctx, g, kv, kv_stride, count, lo, hi, q, scale, quant_query, out, nullptr, 0);
}

int nd_attend_step_i8_noalloc(nd_ctx *ctx, const nd_kv_geom *g, const void *kv, size_t kv_stride,
                              size_t count, const int32_t *lo, const int32_t *hi, const float *q,
                              float scale, int quant_query, float *out)
{
    if (!ctx) return nd::fail(ND_ERR_ARG, "null context");
    float *p = ctx->device >= 0 && ctx->device < kMaxDevices ? g_scratch[ctx->device] : nullptr;
    if (!p) return nd::fail(ND_ERR_HIP, "no-allocation scratch of device %d was not set up",
                            ctx->device);
    // Every partial the merge reads is written by the same call first, so
    // the array's previous contents never matter and nothing is cleared.
    return attend_i8(ctx, g, kv, kv_stride, count, lo, hi, q, scale, quant_query, out, p,
                     kNoAllocScratchFloats);
}

}  // extern "C"
