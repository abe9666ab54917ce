// q4_gemm.hip — matmul_q4_0_dequant (ops/matmul/q4_0.rs:94-181) for more than
// a few rows: raw GGUF Q4_0 blocks times f32 activation rows on the bf16
// matrix cores, without giving up any bit of the f32 activations.
//
//   out[m, n] = sum_b d[n, b] * sum_{k in block b} x[m, k] * (nib[n, k] - 8)
//
// An f32 value is exactly the sum of three bf16 values (q4_common.hpp).  A
// quant (-8 .. 7) is a bf16 value too,
// so every product of the three planes with the quants is exact, and
// v_mfma_f32_16x16x32_bf16 adds them in f32: three MFMAs a block (smallest
// plane first), then one FMA with the block's scale.  Infinities and NaNs
// give NaN, as the regrouped sums of the other Q4_0 kernels do.  Bits below
// 2^-133, which bf16 does not hold, are seen while splitting (values below
// 2^-109 can have them); a workgroup that met any goes over its K again with
// those bits alone, 2^64 times them, and its scales 2^-64 times.
//
// A workgroup computes BM rows x BN channels.  A stage is KB blocks of K:
// its f32 activations and quant bytes are loaded into registers one stage
// ahead, split / unpacked once for the whole workgroup and written to one of
// two LDS buffers, so the product loop has one barrier a stage.  LDS rows are
// 64 bytes (32 bf16) with their 16-byte pieces XOR-swizzled by the row, which
// makes the 16-row fragment reads conflict-free.
//
// Bound: the three MFMAs (1536 cycles a SIMD and block of a 128 x 256 tile)
// and the splitting, unpacking and folding (as many VALU cycles: 43 and 44 % of
// the kernel's, by the counters, where there is a workgroup), which
// the barrier keeps apart: 256 x 4096 x 11008 takes 88 us (263 TFLOP/s of
// f32 products, 0.79 PFLOP/s of bf16 ones); the kernel before it, one wave a
// weight row on the f32 VALU, took 3693 us.  Loading two stages ahead instead
// of one took 5-15 % off; scheduling the splitting among the MFMAs (no branch
// before it) changed nothing for the 8-wave tiles and spilled the 16-wave
// ones.  Error against 64 bits 1.7e-7 (3.1e-7 before).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "q4_common.hpp"

namespace mri {
namespace {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));
struct __attribute__((packed, aligned(2))) U32a2 {
    unsigned v;
};

constexpr int kXcds = 8;

// A barrier that waits for the wave's LDS accesses only.
__device__ inline void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");
}

// Byte of 16-byte piece g of row r in a 64-byte-pitch LDS tile.
__device__ inline int swz(int r, int g) { return r * 64 + ((g ^ ((r >> 1) & 3)) << 4); }

// The end of K part p of np, in blocks: even, so that every tile's stages end
// there too (but for the last part's).
__device__ inline int part_end(int nb, int p, int np) {
    return min(2 * ((nb + 1) / 2 * (p + 1) / np), nb);
}

// The sum is of np K parts (plan_q4), added in part order: by np workgroups a
// tile, which take one each and meet in a workspace, or (TURN) by one, which
// takes them in turn, to the same bits.
template <int BM, int BN, int WM, int WN, int WK, int KB, int PD, bool GG, bool TURN>
__global__ __launch_bounds__(WM *WN *WK * 64, WM * WN * WK > 8 ? 4 : 2) void k_q4_0_gemm(
    const float *__restrict__ x, int M, int K, const uint8_t *__restrict__ w, int N, int n_mt,
    int n_total, int np, int item0, float *__restrict__ out, float *__restrict__ part, int *__restrict__ cnt) {
    constexpr int NT = WM * WN * WK * 64;
    constexpr int RI = BM / 16 / WM, RJ = BN / 16 / WN;  // 16 x 16 sub-tiles of a wave
    constexpr int LA = BM * 8 * KB / NT;                 // float4 pieces a thread
    constexpr int UB = BN * 4 * KB, LB = (UB + NT - 1) / NT;  // 4-byte quant pieces
    constexpr int US = BN * KB, LS = (US + NT - 1) / NT;      // scales
    static_assert(BM % (16 * WM) == 0 && BN % (16 * WN) == 0 && BM * 8 * KB % NT == 0 && KB % WK == 0, "tile");
    static_assert(WK > 1 || KB <= 2, "part_end");
    constexpr int SA = KB * 3 * BM * 64, SB = KB * BN * 64;
    constexpr int STAGE = SA + SB + US * 4;
    extern __shared__ uint4 s_q4[];
    char *lds = reinterpret_cast<char *>(s_q4);

    const int per_xcd = (int)(gridDim.x / kXcds);
    const int item = item0 + (int)(blockIdx.x % kXcds) * per_xcd + (int)(blockIdx.x / kXcds);
    const int ks = TURN ? 1 : np;  // workgroups a tile
    if (item >= n_total * ks) return;
    const int tile = item / ks, kpart = item - tile * ks;
    const int mt = tile % n_mt, nt = tile / n_mt;
    const int t = threadIdx.x, l = t & 63;
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wk = wv / (WM * WN), wm = wv / WN % WM, wn = wv % WN;
    const int nb = K / 32;
    // the stages of K part q are [first(q), first(q + 1))
    auto first = [&](int q) __attribute__((always_inline)) {
        return q == 0 ? 0 : q == np ? (nb + KB - 1) / KB : part_end(nb, q - 1, np) / KB;
    };

    // this thread's pieces of a stage: rows past M and channels past N read
    // the last one (their outputs are not stored); blocks past the end of K
    // read the last block and count as zeros
    const float *a_src[LA];
    int a_kb[LA], a_dst[LA];
#pragma unroll
    for (int i = 0; i < LA; ++i) {
        const int u = t + NT * i, k4 = u % (8 * KB), r = u / (8 * KB);
        a_src[i] = x + (size_t)min(BM * mt + r, M - 1) * K + 4 * (k4 & 7);
        a_kb[i] = k4 >> 3;
        a_dst[i] = (k4 >> 3) * 3 * BM * 64 + swz(r, (k4 & 7) >> 1) + 8 * (k4 & 1);
    }
    const size_t row_bytes = (size_t)nb * kQ4Bytes;
    const uint8_t *b_src[LB];
    int b_kb[LB], b_dst[LB];
#pragma unroll
    for (int i = 0; i < LB; ++i) {
        const int u = min(t + NT * i, UB - 1), g = u & 3, kb = (u >> 2) % KB, n = (u >> 2) / KB;
        b_src[i] = w + (size_t)min(BN * nt + n, N - 1) * row_bytes + 2 + 4 * g;
        b_kb[i] = kb;
        b_dst[i] = SA + kb * BN * 64 + (GG ? swz(n, g >> 1) + 8 * (g & 1) : swz(n, g));
    }
    const uint8_t *s_src[LS];
    int s_kb[LS], s_dst[LS];
#pragma unroll
    for (int i = 0; i < LS; ++i) {
        const int u = min(t + NT * i, US - 1), kb = u % KB, n = u / KB;
        s_src[i] = w + (size_t)min(BN * nt + n, N - 1) * row_bytes;
        s_kb[i] = kb;
        s_dst[i] = SA + SB + (kb * BN + n) * 4;
    }

    struct Regs {
        float4 a[LA];
        unsigned b[LB];
        unsigned s[LS];
    } regs[PD];
    auto load = [&](int s, Regs &r, int s1) __attribute__((always_inline)) {
        const int b0 = min(s, s1 - 1) * KB;
#pragma unroll
        for (int i = 0; i < LA; ++i)
            r.a[i] = *reinterpret_cast<const float4 *>(a_src[i] + 32 * min(b0 + a_kb[i], nb - 1));
#pragma unroll
        for (int i = 0; i < LB; ++i)
            r.b[i] = reinterpret_cast<const U32a2 *>(b_src[i] +
                                                    kQ4Bytes * min(b0 + b_kb[i], nb - 1))->v;
#pragma unroll
        for (int i = 0; i < LS; ++i)
            r.s[i] = *reinterpret_cast<const uint16_t *>(s_src[i] +
                                                        kQ4Bytes * min(b0 + s_kb[i], nb - 1));
    };
    // REST: of the bits that the planes do not hold (q4_rest); otherwise their
    // presence is left in the low half of `lost`.
    unsigned lost = 0;
    auto store = [&](int s, const Regs &r, int s0, auto rest) __attribute__((always_inline)) {
        constexpr bool REST = decltype(rest)::value;
        char *buf = lds + ((s - s0) & 1) * STAGE;
        const int b0 = s * KB;
#pragma unroll
        for (int i = 0; i < LA; ++i) {
            float v[4] = {r.a[i].x, r.a[i].y, r.a[i].z, r.a[i].w};
            if (KB > 1 && b0 + a_kb[i] >= nb) v[0] = v[1] = v[2] = v[3] = 0.0f;
            float md[4], lo[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (REST) v[e] = q4_rest(v[e]);
                md[e] = v[e] - q4_cut(v[e]);
                lo[e] = md[e] - q4_cut(md[e]);
                if constexpr (!REST) lost |= __float_as_uint(lo[e]);
            }
            char *p = buf + a_dst[i];
            *reinterpret_cast<uint2 *>(p) = uint2{q4_top16(v[0], v[1]), q4_top16(v[2], v[3])};
            *reinterpret_cast<uint2 *>(p + BM * 64) =
                uint2{q4_top16(md[0], md[1]), q4_top16(md[2], md[3])};
            *reinterpret_cast<uint2 *>(p + 2 * BM * 64) =
                uint2{q4_top16(lo[0], lo[1]), q4_top16(lo[2], lo[3])};
        }
#pragma unroll
        for (int i = 0; i < LB; ++i) {
            if (UB % NT && t + NT * i >= UB) continue;
            float lo[4], hi[4];
            q4_quants(r.b[i], lo, hi);
            char *p = buf + b_dst[i];
            if constexpr (GG) {  // low nibbles: elements 4g ..; high: 16 + 4g ..
                *reinterpret_cast<uint2 *>(p) = uint2{q4_top16(lo[0], lo[1]), q4_top16(lo[2], lo[3])};
                // piece g / 2 + 2: the swizzle's other half
                const int n = (min(t + NT * i, UB - 1) >> 2) / KB;
                const int g = t & 3;
                *reinterpret_cast<uint2 *>(p + swz(n, (g >> 1) + 2) - swz(n, g >> 1)) =
                    uint2{q4_top16(hi[0], hi[1]), q4_top16(hi[2], hi[3])};
            } else {
                *reinterpret_cast<u4 *>(p) =
                    u4{q4_top16(lo[0], hi[0]), q4_top16(lo[1], hi[1]),
                       q4_top16(lo[2], hi[2]), q4_top16(lo[3], hi[3])};
            }
        }
#pragma unroll
        for (int i = 0; i < LS; ++i) {
            if (US % NT && t + NT * i >= US) continue;
            float d = f16_bits_to_f32(r.s[i]);
            if constexpr (REST) d = q4_rest_scale(d);
            *reinterpret_cast<float *>(buf + s_dst[i]) = KB > 1 && b0 + s_kb[i] >= nb ? 0.0f : d;
        }
    };

    f4 fs[RI][RJ];
#pragma unroll
    for (int i = 0; i < RI; ++i)
#pragma unroll
        for (int j = 0; j < RJ; ++j) fs[i][j] = f4{0, 0, 0, 0};
    const int fr = l & 15, fg = l >> 4;
    const int a_off = swz(wm * RI * 16 + fr, fg);  // + 1024 per 16 rows (swz has period 8)
    const int b_off = SA + swz(wn * RJ * 16 + fr, fg);
    const int d_off = SA + SB + (wn * RJ * 16 + fr) * 4;

    auto product = [&](int s, int s0) __attribute__((always_inline)) {
        const char *buf = lds + ((s - s0) & 1) * STAGE;
#pragma unroll
        for (int k = 0; k < KB / WK; ++k) {
            const int kb = wk * (KB / WK) + k;
            bf8 b[RJ];
            float d[RJ];
#pragma unroll
            for (int j = 0; j < RJ; ++j) {
                b[j] = *reinterpret_cast<const bf8 *>(buf + b_off + kb * BN * 64 + j * 1024);
                d[j] = *reinterpret_cast<const float *>(buf + d_off + (kb * BN + 16 * j) * 4);
            }
            f4 acc[RI][RJ];
#pragma unroll
            for (int p = 2; p >= 0; --p) {
                bf8 a[RI];
#pragma unroll
                for (int i = 0; i < RI; ++i)
                    a[i] = *reinterpret_cast<const bf8 *>(buf + a_off + (kb * 3 + p) * BM * 64 +
                                                          i * 1024);
#pragma unroll
                for (int i = 0; i < RI; ++i)
#pragma unroll
                    for (int j = 0; j < RJ; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            a[i], b[j], p == 2 ? f4{0, 0, 0, 0} : acc[i][j], 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < RI; ++i)
#pragma unroll
                for (int j = 0; j < RJ; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        fs[i][j][e] = __builtin_fmaf(acc[i][j][e], d[j], fs[i][j][e]);
        }
    };
    // K split: this workgroup's slot of the workspace (see below)
    auto put = [&]() __attribute__((always_inline)) {
        constexpr int W = RI * RJ * 4;
        float *mine = part + ((size_t)tile * np + kpart) * (BM * BN) + (size_t)wv * W * 64 + l;
#pragma unroll
        for (int i = 0; i < RI; ++i)
#pragma unroll
            for (int j = 0; j < RJ; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    __hip_atomic_store(mine + ((i * RJ + j) * 4 + e) * 64, fs[i][j][e],
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    };
    const bool split = !TURN && WK == 1 && np > 1;
    __shared__ int s_lost[NT / 64];
    [[maybe_unused]] f4 tot[RI][RJ];  // TURN: the parts so far
    // Stage s lives in register set (s - s0) % PD until it is written to LDS.
    // The barrier waits for LDS only: the loads of the next PD stages stay
    // in flight across it.
    for (int p = kpart;;) {
        const int s0 = first(p), s1 = first(p + 1);
#pragma unroll
        for (int u = 0; u < PD; ++u) load(s0 + u, regs[u], s1);
        store(s0, regs[0], s0, std::false_type{});
        load(s0 + PD, regs[0], s1);
        for (int s = s0; s < s1; s += PD) {
#pragma unroll
            for (int u = 0; u < PD; ++u) {
                if (s + u >= s1) break;
                lds_barrier();
                product(s + u, s0);
                if (s + u + 1 < s1) {
                    store(s + u + 1, regs[(u + 1) % PD], s0, std::false_type{});
                    load(s + u + 1 + PD, regs[(u + 1) % PD], s1);
                }
            }
        }
        // (the next write of a flag is a barrier or more away)
        const bool mine = __any(lost & 0xFFFFu);
        if (l == 0) s_lost[wv] = mine;
        if (split) put();
        lds_barrier();
        if (__any(s_lost[min(l, NT / 64 - 1)])) {
            // rare, so not pipelined: a second pipelined loop, or one loop for
            // both with a branch in store(), cost every call 3-12 %; this 0-1
            for (int s = s0; s < s1; ++s) {
                load(s, regs[0], s1);
                store(s, regs[0], s, std::true_type{});
                lds_barrier();
                product(s, s);
                lds_barrier();
            }
            lost = 0;
            if (split) {
                put();
                lds_barrier();
            }
        }
        if constexpr (!TURN) break;
#pragma unroll
        for (int i = 0; i < RI; ++i)
#pragma unroll
            for (int j = 0; j < RJ; ++j) {
                tot[i][j] = p ? tot[i][j] + fs[i][j] : fs[i][j];
                fs[i][j] = f4{0, 0, 0, 0};
            }
        if (++p == np) break;
    }
    if constexpr (TURN) {
#pragma unroll
        for (int i = 0; i < RI; ++i)
#pragma unroll
            for (int j = 0; j < RJ; ++j) fs[i][j] = tot[i][j];
    }

    if constexpr (WK > 1) {
        // the wave groups' sums, added in group order
        constexpr int W = RI * RJ * 4;
        static_assert((WK - 1) * BM * BN * 4 <= 2 * STAGE, "LDS of the K groups' sums");
        float *red = reinterpret_cast<float *>(lds) + (wm * WN + wn) * W * 64 + l;
        __syncthreads();
        if (wk > 0) {
#pragma unroll
            for (int i = 0; i < W; ++i)
                red[(wk - 1) * BM * BN + i * 64] = fs[i / 4 / RJ][i / 4 % RJ][i % 4];
        }
        __syncthreads();
        if (wk > 0) return;  // (never with np > 1, whose barriers follow)
#pragma unroll
        for (int p = 0; p < WK - 1; ++p)
#pragma unroll
            for (int i = 0; i < W; ++i)
                fs[i / 4 / RJ][i / 4 % RJ][i % 4] += red[p * BM * BN + i * 64];
    }
    if (split) {
        // K split: every part leaves its sums in its slot and counts itself
        // on the tile's counter; the last to arrive adds the parts in part
        // order.  Slots are written with device-scope stores, complete at
        // vmcnt(0) before the barrier and the count, and read with
        // device-scope loads.
        __shared__ int s_last;
        constexpr int W = RI * RJ * 4;
        if (t == 0)
            s_last = __hip_atomic_fetch_add(&cnt[tile], 1, __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT) == np - 1;
        __syncthreads();
        if (!s_last) return;
        f4 tot[RI][RJ];
        for (int p = 0; p < np; ++p) {
            const float *src = part + ((size_t)tile * np + p) * (BM * BN) + (size_t)wv * W * 64 + l;
#pragma unroll
            for (int i = 0; i < RI; ++i)
#pragma unroll
                for (int j = 0; j < RJ; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float v = __hip_atomic_load(src + ((i * RJ + j) * 4 + e) * 64,
                                                          __ATOMIC_RELAXED,
                                                          __HIP_MEMORY_SCOPE_AGENT);
                        tot[i][j][e] = p == 0 ? v : tot[i][j][e] + v;
                    }
        }
#pragma unroll
        for (int i = 0; i < RI; ++i)
#pragma unroll
            for (int j = 0; j < RJ; ++j) fs[i][j] = tot[i][j];
        if (t == 0)  // ready for the next call on this stream
            __hip_atomic_store(&cnt[tile], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // register e of sub-tile (i, j): row 16 i + 4 fg + e, channel 16 j + fr
#pragma unroll
    for (int j = 0; j < RJ; ++j) {
        const int n = BN * nt + 16 * (wn * RJ + j) + fr;
        if (n >= N) continue;
#pragma unroll
        for (int i = 0; i < RI; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = BM * mt + 16 * (wm * RI + i) + 4 * fg + e;
                if (m < M) out[(size_t)m * N + n] = fs[i][j][e];
            }
    }
}

template <int BM, int BN, int WM, int WN, int WK, int KB, int PD, bool GG, bool TURN = false>
mri_status launch_cfg(const float *x, size_t m, size_t k, const uint8_t *w, size_t n, int np,
                      float *out, void *ws, hipStream_t s) {
    const int ks = TURN ? 1 : np;
    constexpr int lds = 2 * (KB * 3 * BM * 64 + KB * BN * 64 + BN * KB * 4);
    auto kernel = &k_q4_0_gemm<BM, BN, WM, WN, WK, KB, PD, GG, TURN>;
    static DeviceOnce attr;
    MRI_HIP(attr.run([&](int) {
        return hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    }));
    const size_t n_mt = (m + BM - 1) / BM, total = n_mt * ((n + BN - 1) / BN);
    const size_t grid = (total * ks + kXcds - 1) / kXcds * kXcds;
    int *cnt = static_cast<int *>(ws);
    float *part = ws ? reinterpret_cast<float *>(cnt + kGemmWsCounters) : nullptr;
    constexpr int threads = WM * WN * WK * 64;
    for (size_t i = 0; i < grid; i += q4_max_grid(threads)) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)std::min(grid - i, q4_max_grid(threads))),
                           dim3(threads), lds, s, x, (int)m, (int)k, w, (int)n, (int)n_mt,
                           (int)total, np, (int)i, out, part, cnt);
        MRI_LAUNCHED("k_q4_0_gemm");
    }
    return MRI_OK;
}

// The tiles for more than 32 rows, and what they cost: the time of one block
// of K with one workgroup on the CU, and of a K part's sums (written and read
// back), in 0.01 us, measured at K = 4096 with 256-11008 channels.
struct Tile {
    int bm, bn, block, part;
    size_t count(size_t m, size_t n) const { return ((m + bm - 1) / bm) * ((n + bn - 1) / bn); }
};
constexpr Tile kTiles[] = {{64, 128, 55, 200}, {128, 128, 81, 350}, {128, 256, 117, 700}};
constexpr int kMaxParts = 8, kMinPartBlocks = 8;

// The tile and K split of least modelled time: passes of the CUs, times the
// blocks of a part, plus the parts.  At 256 x 4096 x 11008 it takes 128 x 256
// tiles in two parts (172 workgroups, one pass), at 512 x 4096 x 4096
// 128 x 128 in two.  The parts belong to the result (their sums are added in
// part order), so they depend on the sizes alone; *whole is the better of the
// first two tiles for one workgroup that takes all parts (the third one's
// registers do not hold their totals too: 333 x 4096 x 12288 430 us, in
// 128 x 128 tiles 215; split 133).
void plan_q4(size_t m, size_t k, size_t n, int *tile, int *parts, int *whole) {
    const long long nb = (long long)(k / 32), cus = std::max(device_cus(), 1);
    long long best = -1, best_whole = -1;
    for (int c = 0; c < 3; ++c) {
        const Tile &tl = kTiles[c];
        const long long tiles = (long long)tl.count(m, n);
        for (int ks = 1; ks <= kMaxParts; ++ks) {
            if (ks > 1 && (nb / ks < kMinPartBlocks || tiles > kGemmWsCounters ||
                           tiles * ks > 4 * cus))
                break;
            const long long passes = (tiles * ks + cus - 1) / cus;
            const long long cost =
                passes * ((nb + ks - 1) / ks) * tl.block + (ks > 1 ? ks * tl.part : 0);
            if (best < 0 || cost < best) best = cost, *tile = c, *parts = ks;
            if (ks == 1 && c < 2 && (best_whole < 0 || cost < best_whole)) best_whole = cost, *whole = c;
        }
    }
}

template <bool GG>
mri_status launch_gemm(const float *x, size_t m, size_t k, const uint8_t *w, size_t n, float *out,
                       hipStream_t s) {
    // Up to 32 rows the K split stays inside the workgroup (WK groups of
    // waves, each its blocks of every stage): nothing is allocated.  Few
    // channels take narrow tiles, which put more workgroups on the chip
    // (16 x 4096 x 4096: 16-channel tiles 10.6 us, 64-channel 18.7; 16 x 4096
    // x 11008: 26.3 and 20.0, the narrow tiles re-reading the activations
    // 688 times).
    const size_t cus = (size_t)std::max(device_cus(), 1);
    if (m <= 16) {
        if ((n + 15) / 16 <= cus + cus / 2)
            return launch_cfg<16, 16, 1, 1, 16, 16, 2, GG>(x, m, k, w, n, 1, out, nullptr, s);
        return launch_cfg<16, 64, 1, 4, 4, 8, 2, GG>(x, m, k, w, n, 1, out, nullptr, s);
    }
    if (m <= 32) {
        if ((n + 31) / 32 <= cus)  // 30 x 4096 x 4096: 19.3 us (64 channels: 27.1)
            return launch_cfg<32, 32, 1, 2, 8, 8, 2, GG>(x, m, k, w, n, 1, out, nullptr, s);
        return launch_cfg<32, 64, 1, 4, 4, 4, 3, GG>(x, m, k, w, n, 1, out, nullptr, s);
    }
    int tile = 0, parts = 1, whole = 0;
    plan_q4(m, k, n, &tile, &parts, &whole);
    if (parts > 1) {
        // A stream that is being captured gets no K split over workgroups: no
        // recorded graph holds the workspace, which may therefore grow at any
        // later call.  One workgroup a tile adds the same parts instead (split
        // and not: 256 x 4096 x 11008 88 and 107 us, 64 x 4096 x 4096 19 and 77).
        void *ws = nullptr;
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(s, &cap) != hipSuccess) {
            (void)hipGetLastError();
            cap = hipStreamCaptureStatusActive;
        }
        if (cap == hipStreamCaptureStatusNone) {
            const Tile &tl = kTiles[tile];
            const mri_status st =
                q4_ws_get(s, kGemmWsCounters * sizeof(int) +
                                 tl.count(m, n) * parts * tl.bm * tl.bn * sizeof(float), &ws);
            if (st) return st;
        }
        switch (ws ? tile : whole + 3) {
        case 0: return launch_cfg<64, 128, 2, 4, 1, 2, 2, GG>(x, m, k, w, n, parts, out, ws, s);
        case 1: return launch_cfg<128, 128, 4, 4, 1, 1, 2, GG>(x, m, k, w, n, parts, out, ws, s);
        case 2: return launch_cfg<128, 256, 2, 8, 1, 1, 2, GG>(x, m, k, w, n, parts, out, ws, s);
        case 3: return launch_cfg<64, 128, 2, 4, 1, 2, 2, GG, true>(x, m, k, w, n, parts, out, ws, s);
        default: return launch_cfg<128, 128, 4, 4, 1, 1, 2, GG, true>(x, m, k, w, n, parts, out, ws, s);
        }
    }
    switch (tile) {
    case 0: return launch_cfg<64, 128, 2, 4, 1, 2, 2, GG>(x, m, k, w, n, 1, out, nullptr, s);
    case 1: return launch_cfg<128, 128, 4, 4, 1, 1, 2, GG>(x, m, k, w, n, 1, out, nullptr, s);
    default: return launch_cfg<128, 256, 2, 8, 1, 1, 2, GG>(x, m, k, w, n, 1, out, nullptr, s);
    }
}

}  // namespace

mri_status launch_q4_gemm(const float *x, size_t m, size_t k, const uint8_t *w, size_t n_out,
                          bool ggml_order, float *out, hipStream_t s) {
    constexpr size_t lim = INT_MAX - 512;
    if (m > lim || k > lim || n_out > lim)
        return set_error(MRI_ERR_UNSUPPORTED, "matmul_q4_0_dequant: a dimension past 2^31");
    return ggml_order ? launch_gemm<true>(x, m, k, w, n_out, out, s)
                      : launch_gemm<false>(x, m, k, w, n_out, out, s);
}

}  // namespace mri
