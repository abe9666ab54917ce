// q4_0.hip — W4A32 Q4_0 products of up to 4 rows on raw GGUF Q4_0 bytes
// (matmul_q4_0_dequant, ops/matmul/q4_0.rs:94-181); more rows go to
// q4_gemm.hip.
//
// The reference dequantizes each block (w = d * (nibble - 8), interleaved
// nibble order: element 2i = low nibble of byte i, 2i+1 = high nibble,
// q4_0.rs:59-68) and accumulates x*w in f32 over K.  Here the sum is
// regrouped per block, which differs from the sequential sum only by rounding
// (the documented 1e-5 * max(|ref|, sum|terms|) contract).
//
// Two forms.
//
// k_q4_0_gemv (1-4 rows, any 2-byte aligned layout): the matrix cores, with
// the f32 activations split exactly into three bf16 planes (q4_common.hpp).
// A workgroup takes 16 channels and its waves split K in laps of 4 blocks:
// lane (r, g) loads block 4 lap + g of channel r, 18 contiguous bytes, and
// holds the block's 32 quants as the B operands of four MFMAs.  All 64 lanes
// hold different k then, so row 4g + p of the A operand carries plane p of
// the activations of block 4 lap + g and is zero elsewhere; the four MFMAs
// add up to register p of lane (r, g) = plane p's sum of its own block, which
// it adds (smallest first) and scales by the d that it loaded.  The planes
// are split once per workgroup into LDS, in parts where K is too long for it;
// bits below 2^-133, which they do not hold, are added in f32 where there are
// any (as in q4_gemm.hip; 0.1-0.25 us a call for seeing that there are none).
// Bound: the unpacking (2.6 VALU
// operations a weight) and its loads, 72-byte pieces of 16 rows.  It took
// 1 x 4128 x 11008 from 23.4 to 10.4 us (the earlier two-lanes-a-block f32
// kernel), 2 x 4128 x 8000 from 33.1 to 9.2 and 4 x 992 x 512 from 12.9 to
// 4.4; against the staged form below 2 x 4096 x 11008 16.8 -> 13.6.  More
// laps in flight, or a wave's laps adjacent, were slower (1 x 4096 x 11008:
// 14-20 us), as was staging the rows through LDS by DMA (12.7-19).
//
// k_q4_0_lds (16-byte aligned weights, K % 256 == 0, so that every row
// starts on 16 bytes; one row, or two): a workgroup takes R consecutive weight rows,
// one contiguous byte range, and moves them to LDS with 16-byte loads (all
// in flight at once); the activations are read from L2.  Lane l of a step
// covers elements 8*(l%4) .. +8 of block l/4 (4 quant
// bytes: low nibble = even element): it reads its 8 activations once and
// applies them to each of the wave's R/4 rows as d * (sum x*nib - 8 * sum x)
// (the activation sum is shared by the rows).  Lane partials are added by a
// wave reduction.
//
// GG (an option without a reference counterpart): upstream GGML's nibble
// order, element i = low nibble of byte i and element i + 16 = its high
// nibble (llama.cpp Q4_0 files).
#include <algorithm>

#include "common.hpp"
#include "q4_common.hpp"

namespace mri {
namespace {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));
struct __attribute__((packed, aligned(4))) Words4 {
    unsigned v[4];
};

constexpr int kThreads = 256;
constexpr int kMaxLds = 160 * 1024;

// LDS of k_q4_0_gemv: [M][3 planes][4 q blocks][64 bytes] and a 16-byte zero
// line, whose place the M * NW * 16 floats of the reduction take, then a flag
// a wave.  The planes of as many laps as it holds (q, a multiple of the waves),
// in parts of about one size.
__host__ __device__ inline size_t q4_gemv_flags(int m, int nw, size_t q) {
    const size_t planes = (size_t)m * 3 * q * 256 + 16, red = (size_t)m * nw * 64;
    return planes > red ? planes : red;
}
size_t q4_gemv_laps(int m, int nw, size_t k) {
    const size_t laps = (k / 32 + 3) / 4;
    const size_t most = (kMaxLds - 16 - 4 * nw) / ((size_t)m * 768);
    if (laps <= most) return laps;
    const size_t parts = (laps + most / nw * nw - 1) / (most / nw * nw);
    return ((laps + parts - 1) / parts + nw - 1) / nw * nw;
}

// PARTS: Q is more laps than LDS holds (qp).
template <int M, int NW, bool PARTS, bool GG>
__global__ __launch_bounds__(NW * 64) void k_q4_0_gemv(const float *__restrict__ x, int K,
                                                       const uint8_t *__restrict__ w, int N,
                                                       int tile0, int qp, float *__restrict__ out) {
    constexpr int NT = NW * 64;
    extern __shared__ u4 s_x[];
    const int t = threadIdx.x, l = t & 63;
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nb = K / 32, Q = (nb + 3) / 4;
    const int r = l & 15, g = l >> 4;
    const int n0 = 16 * (tile0 + (int)blockIdx.x);
    if constexpr (!PARTS) qp = Q;
    const int plane = qp * 16;  // 16-byte pieces
    const int zero = M * 3 * plane;
    // channels past N read the last one (not stored)
    const uint8_t *row = w + (size_t)min(n0 + r, N - 1) * nb * kQ4Bytes;

    // The 18 bytes of this lane's block of a lap (blocks past the end: the
    // last one, counted as zero): the 4-byte aligned words around its quants
    // and, as 2-byte loads that stay inside the block, the last quants and
    // the scale.
    unsigned q[5], d;
    auto load = [&](int lap) __attribute__((always_inline)) {
        const uint8_t *p = row + (size_t)min(4 * lap + g, nb - 1) * kQ4Bytes;
        const Words4 v = *reinterpret_cast<const Words4 *>(((uintptr_t)p + 2) & ~(uintptr_t)3);
#pragma unroll
        for (int i = 0; i < 4; ++i) q[i] = v.v[i];
        q[4] = *reinterpret_cast<const uint16_t *>(p + 16);
        d = *reinterpret_cast<const uint16_t *>(p);
    };
    // Unit u of a row: the 8 activations of word j = u % 4 (4 quant bytes) of
    // block u / 4; LDS holds them in the word's nibble order, low nibbles
    // first.
    auto get = [&](int m, int u, f4 &a, f4 &b) __attribute__((always_inline)) {
        const int blk = min(u >> 2, nb - 1), j = u & 3;
        const float *p = x + (size_t)m * K + 32 * blk;
        a = *reinterpret_cast<const f4 *>(p + (GG ? 4 * j : 8 * j));
        b = *reinterpret_cast<const f4 *>(p + (GG ? 16 + 4 * j : 8 * j + 4));
    };
    // bits that the planes do not hold leave a trace in the low half of `lost`
    unsigned lost = 0;
    auto put = [&](int m, int u, int u0, f4 a, f4 b) __attribute__((always_inline)) {
        if (u >= 4 * nb) a = b = f4{0, 0, 0, 0};
        f4 lo = GG ? a : f4{a[0], a[2], b[0], b[2]};
        f4 hi = GG ? b : f4{a[1], a[3], b[1], b[3]};
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            s_x[(m * 3 + p) * plane + u - u0] = u4{q4_top16(lo[0], lo[1]), q4_top16(lo[2], lo[3]),
                                              q4_top16(hi[0], hi[1]), q4_top16(hi[2], hi[3])};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (p == 2) lost |= __float_as_uint(lo[e]) | __float_as_uint(hi[e]);
                lo[e] -= q4_cut(lo[e]);
                hi[e] -= q4_cut(hi[e]);
            }
        }
    };
    const int units = 16 * Q;
    int *flag = reinterpret_cast<int *>(s_x) + q4_gemv_flags(M, NW, qp) / 4;
    float acc[M];
#pragma unroll
    for (int m = 0; m < M; ++m) acc[m] = 0.0f;
    const bool on = (r >> 2) == g && (r & 3) < 3;
    const int st = on ? 1 : 0;
    f4 xa[M], xb[M];
#pragma unroll
    for (int m = 0; m < M; ++m) get(m, min(t, units - 1), xa[m], xb[m]);
    load(wv);
    if (t == 0) s_x[zero] = u4{0, 0, 0, 0};
#pragma unroll
    for (int m = 0; m < M; ++m)
        if (t < 16 * qp) put(m, t, 0, xa[m], xb[m]);
    for (int q0 = 0;;) {
        const int q1 = PARTS ? min(q0 + qp, Q) : Q;
        if (q0)  // the last part's planes are read
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");
        for (int u = q0 ? 16 * q0 + t : t + NT; u < 16 * q1; u += NT) {
#pragma unroll
            for (int m = 0; m < M; ++m) {
                f4 a, b;
                get(m, u, a, b);
                put(m, u, 16 * q0, a, b);
            }
        }
        // LDS only: the weight loads stay in flight
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");

        for (int lap = q0 + wv; lap < q1; lap += NW) {
            const int blk = 4 * lap + g;
            const float ds = blk < nb ? f16_bits_to_f32(d) : 0.0f;
            // quants at 2 bytes past a word: shifted into place
            const uintptr_t p = (uintptr_t)row + (uintptr_t)(min(blk, nb - 1) * (size_t)kQ4Bytes);
            const unsigned sh = 2u - ((unsigned)p & 2u);
            bf8 b[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float lo[4], hi[4];
                q4_quants(__builtin_amdgcn_alignbyte(q[j + 1], q[j], sh), lo, hi);
                b[j] = __builtin_bit_cast(
                    bf8, u4{q4_top16(lo[0], lo[1]), q4_top16(lo[2], lo[3]), q4_top16(hi[0], hi[1]),
                            q4_top16(hi[2], hi[3])});
            }
            load(lap + NW);
#pragma unroll
            for (int m = 0; m < M; ++m) {
                f4 c{0, 0, 0, 0};
                const int ai = on ? (m * 3 + (r & 3)) * plane + 4 * g + 16 * (lap - q0) : zero;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf8, s_x[ai + st * j]), b[j], c, 0, 0, 0);
                acc[m] = __builtin_fmaf((c[2] + c[1]) + c[0], ds, acc[m]);
            }
        }
        q0 += qp;
        if (!PARTS || q0 >= Q) break;
    }
    // the four lane groups' blocks, then the waves' laps in wave order
    auto finish = [&]() __attribute__((always_inline)) {
        float *red = reinterpret_cast<float *>(s_x);
#pragma unroll
        for (int m = 0; m < M; ++m) {
            float s = acc[m] + __shfl_xor(acc[m], 16);
            s += __shfl_xor(s, 32);
            if (l < 16) red[(m * NW + wv) * 16 + l] = s;
        }
        __syncthreads();
        const int any = flag[min(l, NW - 1)];
        if (t < 16 * M) {
            const int m = t >> 4, n = n0 + (t & 15);
            float s = red[m * NW * 16 + (t & 15)];
#pragma unroll
            for (int v = 1; v < NW; ++v) s += red[(m * NW + v) * 16 + (t & 15)];
            if (n < N) out[(size_t)m * N + n] = s;
        }
        return any;
    };
    const bool mine = __any(lost & 0xFFFFu);
    if (l == 0) flag[wv] = mine;
    __syncthreads();
    if (__builtin_expect(!__any(finish()), 1)) return;
    // rare: the lost bits' products (q4_rest) in f32, lane (r, g)'s of channel
    // r and every (4 NW)-th block
#pragma unroll 1
    for (int b = t >> 4; b < nb; b += NT / 16) {
        const uint8_t *p = row + (size_t)b * kQ4Bytes;
        const float ds =
            q4_rest_scale(f16_bits_to_f32(*reinterpret_cast<const uint16_t *>(p)));
        float c[M] = {};
#pragma unroll 1
        for (int e = 0; e < 32; ++e) {
            const int nib = GG ? p[2 + (e & 15)] >> (e >> 4) * 4 : p[2 + (e >> 1)] >> (e & 1) * 4;
#pragma unroll
            for (int m = 0; m < M; ++m)
                c[m] = __builtin_fmaf(q4_rest(x[(size_t)m * K + 32 * b + e]),
                                      (float)((nib & 15) - 8), c[m]);
        }
#pragma unroll
        for (int m = 0; m < M; ++m) acc[m] = __builtin_fmaf(c[m], ds, acc[m]);
    }
    __syncthreads();
    finish();
}

__global__ __launch_bounds__(kThreads) void k_zero(size_t n, unsigned *__restrict__ p) {
    for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n;
         i += (size_t)gridDim.x * kThreads)
        p[i] = 0;
}

template <int R, int M, bool GG>
__global__ __launch_bounds__(kThreads) void k_q4_0_lds(const float *__restrict__ x, int K,
                                                       const uint8_t *__restrict__ w, int N,
                                                       size_t pitch, float *__restrict__ out) {
    constexpr int RW = R / 4;  // rows per wave
    extern __shared__ int4 s_raw[];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int nb = K / 32, row_bytes = nb * kQ4Bytes;
    const int n0 = blockIdx.x * R, rows = min(R, N - n0);
    const uint8_t *s_w = reinterpret_cast<const uint8_t *>(s_raw);
    {
        // every load in flight before the first store (at most 12 pieces a
        // thread: the launcher keeps R rows within 48 KiB; the pieces past
        // the rows re-read the last one, which measured faster than
        // skipping them under a branch: 11.8 against 21.3 us at N = 11008)
        const int4 *src = reinterpret_cast<const int4 *>(w + (size_t)n0 * row_bytes);
        const int n16 = rows * row_bytes / 16;
        int4 v[12];
#pragma unroll
        for (int u = 0; u < 12; ++u) v[u] = src[min(t + kThreads * u, n16 - 1)];  // n16 >= 1
#pragma unroll
        for (int u = 0; u < 12; ++u) {
            const int i = t + kThreads * u;
            if (i < n16) s_raw[i] = v[u];
        }
    }
    __syncthreads();
    const int steps = (nb * 4 + 63) / 64;
    // rows past `rows` read stale LDS and are never stored
    float acc[M][RW] = {};
    for (int st = 0; st < steps; ++st) {
        const int idx = st * 64 + lane, p = idx & 3;
        const bool ok = (idx >> 2) < nb;
        const int b = ok ? idx >> 2 : nb - 1;
        float4 xa[M], xb[M];
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const float4 *xv =
                reinterpret_cast<const float4 *>(x + (size_t)m * K + 32 * b + 8 * p);
            xa[m] = xv[0], xb[m] = xv[1];
            if (!ok) xa[m] = xb[m] = float4{0, 0, 0, 0};
        }
        float dq[RW];
        unsigned lo[RW], hi[RW];
#pragma unroll
        for (int r = 0; r < RW; ++r) {
            const uint8_t *blk = s_w + (size_t)(wv * RW + r) * row_bytes + b * kQ4Bytes;
            dq[r] = f16_bits_to_f32(*reinterpret_cast<const uint16_t *>(blk));
            if constexpr (GG) {
                // elements 8p .. 8p+7: nibble p / 2 of bytes 8 (p % 2) .. +7,
                // regrouped into the (even, odd) element words below
                const uint16_t *qs = reinterpret_cast<const uint16_t *>(blk + 2 + 8 * (p & 1));
                const int sh = 4 * (p >> 1);
                const unsigned a0 = ((unsigned)qs[0] | ((unsigned)qs[1] << 16)) >> sh;
                const unsigned a1 = ((unsigned)qs[2] | ((unsigned)qs[3] << 16)) >> sh;
                // a0 bytes = elements 0..3, a1 bytes = elements 4..7
                const unsigned e0 = a0 & 0x0F0F0F0Fu, e1 = a1 & 0x0F0F0F0Fu;
                lo[r] = (e0 & 0xFFu) | ((e0 >> 8) & 0xFF00u) | ((e1 << 16) & 0xFF0000u) |
                        ((e1 << 8) & 0xFF000000u);          // elements 0, 2, 4, 6
                hi[r] = ((e0 >> 8) & 0xFFu) | ((e0 >> 16) & 0xFF00u) |
                        ((e1 << 8) & 0xFF0000u) | (e1 & 0xFF000000u);  // 1, 3, 5, 7
            } else {
                const unsigned q =
                    (unsigned)*reinterpret_cast<const uint16_t *>(blk + 2 + 4 * p) |
                    ((unsigned)*reinterpret_cast<const uint16_t *>(blk + 4 + 4 * p) << 16);
                lo[r] = q & 0x0F0F0F0Fu;          // elements 0, 2, 4, 6 (low nibbles)
                hi[r] = (q >> 4) & 0x0F0F0F0Fu;   // elements 1, 3, 5, 7
            }
            // opaque, so that each nibble is one v_cvt_f32_ubyte of its byte
            // and not a field extraction too (1 x 4096 x 11008 12.1 -> 11.8 us
            // a call, the same bits; aligned 8-byte LDS reads of the quants
            // instead of two 2-byte ones were slower, 12.0, unaligned 4-byte
            // ones far slower, 18.2); for one row a wave the extractions are the
            // faster form (1 x 14336 x 6144 24.2 -> 21.0, 12288 x 12288 34.5 ->
            // 31.3)
            if constexpr (RW > 1) asm("" : "+v"(lo[r]), "+v"(hi[r]));
        }
        // d * sum_e x_e * (nib_e - 8) = d * (sum_e x_e * nib_e - 8 * sum_e x_e);
        // the activation sum is shared by the wave's weight rows, and the
        // rows' chains are interleaved
        float xs[M], sn[M][RW];
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const float4 a = xa[m], c = xb[m];
            xs[m] = ((a.x + a.y) + (a.z + a.w)) + ((c.x + c.y) + (c.z + c.w));
        }
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int r = 0; r < RW; ++r) {
                const float q = (float)(((e & 1 ? hi[r] : lo[r]) >> (e >> 1) * 8) & 0xFF);
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    const float4 &h = e < 4 ? xa[m] : xb[m];
                    const float v = (e & 3) == 0 ? h.x : (e & 3) == 1 ? h.y : (e & 3) == 2 ? h.z : h.w;
                    sn[m][r] = e ? fmaf(v, q, sn[m][r]) : v * q;
                }
            }
#pragma unroll
        for (int r = 0; r < RW; ++r)
#pragma unroll
            for (int m = 0; m < M; ++m)
                acc[m][r] = fmaf(dq[r], fmaf(-8.0f, xs[m], sn[m][r]), acc[m][r]);
    }
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int r = 0; r < RW; ++r) {
            float v = acc[m][r];
            for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
            const int row = wv * RW + r;
            if (lane == 0 && row < rows) out[(size_t)m * pitch + n0 + row] = v;
        }
}

size_t q4_lds_bytes(int r, size_t k) { return (size_t)r * (k / 32) * kQ4Bytes; }

template <int R, int M, bool GG>
mri_status launch_lds(const float *x, size_t k, const uint8_t *w, size_t n_out,
                      float *out, hipStream_t s) {
    static DeviceOnce attr;
    MRI_HIP(attr.run([](int) {
        return hipFuncSetAttribute(reinterpret_cast<const void *>(&k_q4_0_lds<R, M, GG>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds);
    }));
    const size_t step = R * q4_max_grid(kThreads);
    for (size_t n = 0; n < n_out; n += step) {
        const size_t c = std::min(n_out - n, step);
        hipLaunchKernelGGL((k_q4_0_lds<R, M, GG>), dim3((unsigned)((c + R - 1) / R)), dim3(kThreads),
                           q4_lds_bytes(R, k), s, x, (int)k, w + n * (k / 32) * kQ4Bytes, (int)c,
                           n_out, out + n);
        MRI_LAUNCHED("k_q4_0_lds");
    }
    return MRI_OK;
}

template <int M, int NW, bool PARTS, bool GG>
mri_status launch_gemv(const float *x, size_t k, const uint8_t *w, size_t n_out, float *out,
                       hipStream_t s) {
    static DeviceOnce attr;
    MRI_HIP(attr.run([](int) {
        return hipFuncSetAttribute(reinterpret_cast<const void *>(&k_q4_0_gemv<M, NW, PARTS, GG>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds);
    }));
    const size_t tiles = (n_out + 15) / 16, step = q4_max_grid(NW * 64);
    const size_t qp = q4_gemv_laps(M, NW, k);
    for (size_t t = 0; t < tiles; t += step) {
        hipLaunchKernelGGL((k_q4_0_gemv<M, NW, PARTS, GG>), dim3((unsigned)std::min(tiles - t, step)),
                           dim3(NW * 64), q4_gemv_flags(M, NW, qp) + 4 * NW, s, x, (int)k, w,
                           (int)n_out, (int)t, (int)qp, out);
        MRI_LAUNCHED("k_q4_0_gemv");
    }
    return MRI_OK;
}

template <int NW, bool PARTS, bool GG>
mri_status launch_gemv_rows(const float *x, size_t m, size_t k, const uint8_t *w, size_t n_out,
                            float *out, hipStream_t s) {
    switch (m) {
    case 1: return launch_gemv<1, NW, PARTS, GG>(x, k, w, n_out, out, s);
    case 2: return launch_gemv<2, NW, PARTS, GG>(x, k, w, n_out, out, s);
    case 3: return launch_gemv<3, NW, PARTS, GG>(x, k, w, n_out, out, s);
    default: return launch_gemv<4, NW, PARTS, GG>(x, k, w, n_out, out, s);
    }
}

template <bool GG>
mri_status launch_q4(const float *x, size_t m, size_t k, const uint8_t *w, size_t n_out,
                     float *out, hipStream_t s) {
    if (k == 0) return launch_zero(out, m * n_out, s);
    const size_t cus = (size_t)std::max(device_cus(), 1), tiles = (n_out + 15) / 16;
    const bool few = 2 * tiles <= 3 * cus;  // 16-channel workgroups fit about one a CU
    // the staged form: 16-byte aligned rows (K % 256 == 0) and operands
    const bool al = ((uintptr_t)w & 15) == 0 && ((uintptr_t)x & 15) == 0 && k % 256 == 0;
    // k_q4_0_gemv is the faster one where its workgroups take half of the CUs
    // to all of them once and K is long, its waves splitting K (us, staged and
    // not: 11008 -> 4096 12.5 and 9.8, -> 2048 9.2 and 9.6, -> 4352 13.6 and
    // 15.6; 8448 -> 4096 10.0 and 8.5), but for K of whole 2048s, where the 16
    // rows of a load start at one place of their lines (8192 -> 4096 9.7 and
    // 10.6, 14336 -> 3072 11.5 and 14.6).
    const bool lines = k % 2048 == 0;
    const bool rows16 = k >= 8192 && 2 * tiles > cus && tiles <= cus && !lines;
    if (al && m == 1 && n_out <= (1u << 30) && !rows16) {
        // rows per workgroup: 8, or 4 where 8 rows exceed ~40 KiB of LDS.
        // Measured at K = 4096 (us per call): 8 rows 11.8 (N = 11008) and
        // 6.4 (N = 4096), against 13.1 and 8.4 for 16 rows and 12.7 and 6.4
        // for 4 (more workgroups per CU overlap one's loads with another's
        // arithmetic; 4 also where long rows are few: 8192 -> 1024 6.5 and 6.9
        // with 8, -> 3072 8.2 and 9.4).  k_q4_0_gemv takes 13.3 and 7.0 there,
        // its 16 channels' loads being 72-byte pieces.
        if (q4_lds_bytes(8, k) <= 40 * 1024 && !(k >= 8192 && tiles <= cus))
            return launch_lds<8, 1, GG>(x, k, w, n_out, out, s);
        if (q4_lds_bytes(4, k) <= 48 * 1024) return launch_lds<4, 1, GG>(x, k, w, n_out, out, s);
    }
    // Two rows, staged, where a line offset costs k_q4_0_gemv more: in its
    // second pass of the CUs (8192 -> 4352 13.6 us, not staged 19.8), and with
    // few workgroups on a long K (14336 -> 2048 12.2 and 16.5).
    if (al && m == 2 && n_out <= (1u << 30) && lines) {
        if (few && tiles > cus && q4_lds_bytes(8, k) <= 48 * 1024)
            return launch_lds<8, 2, GG>(x, k, w, n_out, out, s);
        if (2 * tiles <= cus && k >= 8192 && q4_lds_bytes(4, k) <= 48 * 1024)
            return launch_lds<4, 2, GG>(x, k, w, n_out, out, s);
    }
    // Rows 3 and 4 on many channels go to the tiled kernel, which unpacks
    // each weight once for 16 rows and streams (4 x 4096 x 11008 19.1 us
    // against 23.6; at N = 4096 10.6 against 8.3).  16 waves where a CU has one
    // workgroup: few channels and a long K, or planes that LDS holds in parts
    // (2 x 14336 x 4096 17.2 us, in the tiled kernel 27.8; 2 x 28672 x 8192 57
    // and 114, 8 waves 67).
    if (n_out <= (1u << 30) && k <= (1u << 20) && (m <= 2 || (m <= 4 && few))) {
        const bool wide = k >= 8192 && few;
        if (q4_gemv_laps((int)m, 16, k) < (k / 32 + 3) / 4)
            return launch_gemv_rows<16, true, GG>(x, m, k, w, n_out, out, s);
        return wide ? launch_gemv_rows<16, false, GG>(x, m, k, w, n_out, out, s)
                    : launch_gemv_rows<8, false, GG>(x, m, k, w, n_out, out, s);
    }
    return launch_q4_gemm(x, m, k, w, n_out, GG, out, s);
}

}  // namespace

mri_status launch_zero(void *p, size_t words, hipStream_t s) {
    const size_t grid = std::min<size_t>((words + kThreads - 1) / kThreads, 65536);
    hipLaunchKernelGGL(k_zero, dim3((unsigned)grid), dim3(kThreads), 0, s, words,
                       static_cast<unsigned *>(p));
    MRI_LAUNCHED("k_zero");
    return MRI_OK;
}

mri_status launch_q4_0_dequant(const float *x, size_t m, size_t k, const uint8_t *w,
                               size_t n_out, bool ggml_order, float *out, hipStream_t s) {
    if (m == 0 || n_out == 0) return MRI_OK;
    return ggml_order ? launch_q4<true>(x, m, k, w, n_out, out, s)
                      : launch_q4<false>(x, m, k, w, n_out, out, s);
}

}  // namespace mri
