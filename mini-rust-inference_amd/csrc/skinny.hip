// skinny.hip — quantized matmul on CDNA4 MFMA for INT8 at 5..63 rows and, for
// Q8_0 and W4A8, from 5 rows up to the sizes of the LDS-tiled GEMM (and at
// every row count where the reference's block order is asked for).
//
// The weight stream dominates (M*K activation bytes vs N*K weight bytes), so
// both kernels stream the 1 KiB weight chunks of 16-row tiles
// (INT8: slab-major chunks; Q8_0: the tile's lap blocks, quants and scales
// together), with the activation rows read from a quantized buffer ([M][kp], or
// row groups):
//   * per-channel INT8: v_mfma_i32_16x16x64_i8 accumulates exact int32 dot
//     products for 16 (m) x 16 (n) outputs; the f32 epilogue
//     ((f32)acc * s_a) * s_w runs once at the end (int8.rs:93);
//   * Q8_0: one v_mfma_i32_16x16x32_i8 per 32-element block gives the exact
//     per-block int32 dot; each lane then applies ((f32)dot * s_a[m]) * d[n,b]
//     and adds it to its running f32 sum in block order — the order of
//     q8_direct.rs:269-282, so the f32 result is bit-identical.
// MFMA output mapping (16x16 family): lane l, register i holds row
// (activation) m = 4*(l/16) + i and column (weight row) n = l % 16.
// The M <= 4 decode case uses the K-split kernels of gemv_int8.hip and
// gemv_q8.hip instead.
#include <algorithm>
#include <type_traits>

#include "gemv_common.hpp"

namespace mri {
using namespace gemv;
namespace {

// ---------------------------------------------------------------------------
// Per-channel INT8.  A workgroup takes NT tiles of 16 channels and all rows
// (MT activation tiles of 16); its S waves split K into contiguous runs of
// chunks, each in two register buffers of U chunks, and add their int32 sums
// through LDS (exact in any order), each wave finishing its share of the
// output registers.  One wave a tile, as this kernel had before, left 256
// tiles with one wave a CU and re-read the weights for every 32 rows:
// 24 x 4096 x 4096 8.4 -> 5.4 us, 60 x 4096 x 11008 with its quantization
// 43.4 -> 25.5.
// ---------------------------------------------------------------------------
template <int MT, int NT, int U, int S>
__global__ __launch_bounds__(S * kWave) void k_skinny_int8(
    const int8_t *__restrict__ act, int M, size_t kp,
    const float *__restrict__ sa_ptr, int sa_stride, float sa_value,
    const v4i *__restrict__ tiles, const float *__restrict__ wscales, int N, int n_tiles,
    int P, float *__restrict__ out, int32_t *__restrict__ acc_out) {
    constexpr int E = MT * NT * 4;  // output registers
    extern __shared__ int32_t red[];  // [S][E][kWave]
    const int T0 = blockIdx.x * NT;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l = threadIdx.x & 63;
    const int r = l & 15, g = l >> 4;
    const int lo = split_lo(P, S, wv), hi = split_lo(P, S, wv + 1);
    const int last = hi > 0 ? hi - 1 : 0;             // loads past the run re-read its end
    const size_t pitch = (size_t)n_tiles * kWave;    // slab-major chunks
    const v4i *wp[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)  // tiles past the end read the last (not stored)
        wp[t] = tiles + (size_t)min(T0 + t, n_tiles - 1) * kWave + l;
    const v4i *ap[MT];
    bool aval[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m = mt * 16 + r;
        aval[mt] = m < M;
        ap[mt] = reinterpret_cast<const v4i *>(act + (size_t)(aval[mt] ? m : 0) * kp) + g;
    }
    const v4i zero = {0, 0, 0, 0};
    v4i acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[mt][t] = zero;

    v4i wb[2][NT][U];
    v4i ab[2][MT][U];

    // Loads are unconditional (the chunk index is clamped) and rows m >= M
    // are zeroed at use, so the compiler never has to wait for an older load
    // before a conditional write to the same registers.
    auto load = [&](int buf, int p0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int t = 0; t < NT; ++t)
                wb[buf][t][u] =
                    __builtin_nontemporal_load(wp[t] + (size_t)min(p0 + u, last) * pitch);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                ab[buf][mt][u] = ap[mt][(size_t)min(p0 + u, last) * 4];
    };
    // GUARD: only the last group can run past the end.
    auto compute = [&](int buf, int p0, auto guard) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (!decltype(guard)::value || p0 + u < hi) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const v4i a = aval[mt] ? ab[buf][mt][u] : zero;
#pragma unroll
                    for (int t = 0; t < NT; ++t)
                        acc[mt][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                            a, wb[buf][t][u], acc[mt][t], 0, 0, 0);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    // Two register buffers: while one group of U chunks is consumed the next
    // group's loads are in flight.
    int p = lo;
    load(0, p);
    for (;;) {
        if (p + U >= hi) {
            compute(0, p, std::true_type{});
            break;
        }
        load(1, p + U);
        compute(0, p, std::false_type{});
        p += U;
        if (p + U >= hi) {
            compute(1, p, std::true_type{});
            break;
        }
        load(0, p + U);
        compute(1, p, std::false_type{});
        p += U;
    }
#pragma unroll
    for (int e = 0; e < E; ++e)
        red[(wv * E + e) * kWave + l] = acc[e / 4 / NT][e / 4 % NT][e % 4];
    __syncthreads();

    for (int e = wv; e < E; e += S) {  // register e % 4 of row tile e / 4 / NT
        uint32_t sum = 0;
#pragma unroll
        for (int q = 0; q < S; ++q) sum += (uint32_t)red[(q * E + e) * kWave + l];
        const int m = e / (4 * NT) * 16 + 4 * g + (e & 3);
        const int n = (T0 + e / 4 % NT) * 16 + r;
        if (m < M && n < N) {
            const float sa = sa_ptr ? sa_ptr[(size_t)m * sa_stride] : sa_value;
            float v = (float)(int32_t)sum * sa;
            v = v * wscales[n];
            out[(size_t)m * N + n] = v;
            if (acc_out) acc_out[(size_t)m * N + n] = (int32_t)sum;
        }
    }
}

// ---------------------------------------------------------------------------
// Q8_0: AG groups of 16 activation rows and NT tiles of 16 output channels a
// wave, which sweeps all of K in laps of one scale group (4
// chunks = 8 blocks) and keeps RL laps of loads in flight: per chunk and tile one
// 16-byte load of the weight chunk and, per activation group, one 16-byte
// load of the rows' matching activation bytes (chunk-permuted, so its two
// halves are the A operands of the chunk's two blocks).  Per block and
// group one v_mfma_i32_16x16x32_i8 gives the exact int32 dots of 16 rows x
// 16 channels; each lane then adds ((f32)dot * s_a[m]) * d[n,b] to its
// running sums in block order (q8_direct.rs:269-282), so the f32 result is
// bit-identical.  The sweep has no global memory instruction other than the
// ring's loads and no data-dependent branch, so every wait leaves the
// younger loads in flight.  Rows m >= M read row 0's activations, or in row
// groups what lies in the last group; their results are never stored.
//
// W4 (Q4_0 weights of the W4A8 path): a lap's quants are two 16-byte pieces
// per lane; the 8-byte B operand of block h of chunk c is the u32 word
// 2(c % 2) + h of piece c / 2 with each nibble moved to the high half of its
// byte (16 * quant as int8), and the MFMA result is divided by 16 exactly.
// ---------------------------------------------------------------------------
template <int AG, int NT, int RL, int CS, bool DEBUG, bool W4>
__global__ __launch_bounds__(kWave) void k_skinny_q8_0(
    const int8_t *__restrict__ act, int M, int kp, const float *__restrict__ sa_rows,
    const v4i *__restrict__ laps, int N, int n_tiles, int G, int nb, float *__restrict__ out,
    int32_t *__restrict__ block_dots, int ns, int mg) {
    // wave -> (NT adjacent tiles, set of AG activation groups); the ns waves of
    // the tiles are adjacent, so that the weight chunks they all stream are
    // fetched from HBM once.  With several waves per tile the grid (a multiple
    // of 8) is taken XCD-major: workgroups are dispatched to the 8 XCDs
    // round-robin, and consecutive indices of one XCD share its L2.
    int wv = blockIdx.x;
    if (ns > 1) wv = (int)(blockIdx.x % 8) * (int)(gridDim.x / 8) + (int)(blockIdx.x / 8);
    const int T0 = wv / ns * NT;
    const int a0 = wv % ns * AG;  // first activation group of the wave
    if (T0 >= n_tiles) return;  // whole waves only; the kernel has no barrier
    const int l = threadIdx.x;
    const int r = l & 15, g = l >> 4;
    // a tile's lap blocks: quant piece c of lap q at v4i offset
    // q * LB + c * 64 (+ lane), the lap's scales at q * LB + SO (+ row); tiles
    // past the end read the last one and store nothing
    constexpr size_t LB = (W4 ? kQ4LapBytes : kQ8LapBytes) / 16;
    constexpr int SO = W4 ? 128 : 256;
    constexpr int NP = W4 ? 2 : 4;  // quant pieces per lap and lane
    // (addresses as a wave-uniform base and a 32-bit lane offset, so that no
    // vector instruction goes into them: a wave that is alone on its SIMD is
    // bound by those it issues)
    const char *wp[NT];
    int n[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        wp[t] = reinterpret_cast<const char *>(laps + (size_t)min(T0 + t, n_tiles - 1) * G * LB);
        n[t] = T0 + t < n_tiles ? (T0 + t) * 16 + r : N;
    }
    const unsigned wl = 16 * l, sl = 16 * (SO + r);
    auto at = [](const char *base, unsigned lane) __attribute__((always_inline)) {
        return reinterpret_cast<const v4i *>(base + (size_t)lane);
    };
    // the activations: this lane's 16 bytes of chunk p of its rows at
    // act + p * cs + al[a], in rows (past M: row 0) or in mg row groups.  CS
    // states the stride for one group or rows, where it is known: a lap's four
    // loads then share one address (14 x 12288 x 2560: 4 % of a wave's time).
    unsigned al[AG];
    const size_t cs = CS ? CS : mg ? (size_t)mg * 1024 : 64;
    const char *ap = reinterpret_cast<const char *>(act);
    float sa[AG][4], fs[AG][NT][4];
#pragma unroll
    for (int a = 0; a < AG; ++a) {
        const int m = 16 * (a0 + a) + r;
        al[a] = mg ? 1024u * (unsigned)min(a0 + a, mg - 1) + 64 * r + 16 * g
                   : (unsigned)(m < M ? m : 0) * (unsigned)kp + 16 * g;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            sa[a][i] = sa_rows[min(16 * (a0 + a) + 4 * g + i, M - 1)];
#pragma unroll
            for (int t = 0; t < NT; ++t) fs[a][t][i] = 0.0f;
        }
    }
    v4i wr[RL][NT][4];
    v4i xr[RL][4][AG];
    v4i sr[RL][NT];
#pragma unroll
    for (int u = 0; u < RL; ++u) {
        const int q = min(u, G - 1);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
                if (c < NP)
                    wr[u][t][c] =
                        __builtin_nontemporal_load(at(wp[t] + ((size_t)q * LB + c * 64) * 16, wl));
#pragma unroll
            for (int a = 0; a < AG; ++a) xr[u][c][a] = *at(ap + (size_t)(4 * q + c) * cs, al[a]);
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) sr[u][t] = *at(wp[t] + (size_t)q * LB * 16, sl);
    }
    const v4i zero = {0, 0, 0, 0};
    // Without W4 each block's MFMA starts from the bits of 1.5 * 2^23, so an
    // output register read as f32 is 12582912 + dot exactly (|dot| < 2^22);
    // one full-rate subtract gives (f32)dot, bit for bit what the half-rate
    // v_cvt_f32_i32 gives.
    const v4i cinit = W4 ? zero : v4i{kDotBias, kDotBias, kDotBias, kDotBias};

    // Lap L in ring slot U.  REFILL: lap L + RL exists and is loaded into
    // the slot; CHECK: skip padding blocks past nb (last laps only).
    auto lap = [&](int L, auto slot, bool refill, auto check) __attribute__((always_inline)) {
        constexpr int U = decltype(slot)::value;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            v4i d[2][AG][NT];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    long bv;
                    if constexpr (W4) {
                        const v4i pc = wr[U][t][c >> 1];
                        const int wd = (c & 1) ? (h ? pc.w : pc.z) : (h ? pc.y : pc.x);
                        constexpr int kHi = (int)0xF0F0F0F0u;
                        bv = (long)(((unsigned long)(unsigned)(wd & kHi) << 32) |
                                    (unsigned)((wd << 4) & kHi));
                    } else {
                        bv = h ? hi8(wr[U][t][c]) : lo8(wr[U][t][c]);
                    }
#pragma unroll
                    for (int a = 0; a < AG; ++a) {
                        d[h][a][t] = __builtin_amdgcn_mfma_i32_16x16x32_i8(
                            h ? hi8(xr[U][c][a]) : lo8(xr[U][c][a]), bv, cinit, 0, 0, 0);
                        if constexpr (W4) {
#pragma unroll
                            for (int i = 0; i < 4; ++i) d[h][a][t][i] >>= 4;
                        }
                    }
                }
            }
            if (refill) {
                const size_t p = (size_t)(4 * (L + RL) + c);
                if (!W4 || (c & 1)) {
                    const int pi = W4 ? c >> 1 : c;
#pragma unroll
                    for (int t = 0; t < NT; ++t)
                        wr[U][t][pi] = __builtin_nontemporal_load(
                            at(wp[t] + ((size_t)(L + RL) * LB + pi * 64) * 16, wl));
                }
#pragma unroll
                for (int a = 0; a < AG; ++a) xr[U][c][a] = *at(ap + p * cs, al[a]);
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int b = 8 * L + 2 * c + h;
                if (!decltype(check)::value || b < nb) {
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        const unsigned word = (unsigned)sr[U][t][c];
                        const float ds = f16_bits_to_f32(h ? (word >> 16) : (word & 0xFFFFu));
#pragma unroll
                        for (int a = 0; a < AG; ++a) {
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                const int dv = d[h][a][t][i];
                                float tm = (W4 ? (float)dv : __int_as_float(dv) - kDotBiasF) *
                                           sa[a][i];
                                tm = tm * ds;
                                fs[a][t][i] = fs[a][t][i] + tm;
                            }
                            if constexpr (DEBUG) {
#pragma unroll
                                for (int i = 0; i < 4; ++i) {
                                    const int m = 16 * (a0 + a) + 4 * g + i;
                                    if (m < M && n[t] < N)
                                        block_dots[((size_t)m * N + n[t]) * nb + b] =
                                            W4 ? d[h][a][t][i] : d[h][a][t][i] - kDotBias;
                                }
                            }
                        }
                    }
                }
            }
        }
        if (refill) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
                sr[U][t] = *at(wp[t] + (size_t)(L + RL) * LB * 16, sl);
        }
        // keep the next lap's uses of its (younger) loads below this point
        __builtin_amdgcn_sched_barrier(0);
    };

    using T1 = std::true_type;
    using F0 = std::false_type;
    {
        const int k = G / RL, rem = G - k * RL;
        for (int it = 0; it + 1 < k; ++it)
            static_for<RL>([&](auto u) { lap(it * RL + u, u, true, F0{}); });
        if (k > 0)
            static_for<RL>([&](auto u) { lap((k - 1) * RL + u, u, u < rem, T1{}); });
        static_for<RL>([&](auto u) {
            if (u < rem) lap(k * RL + u, u, false, T1{});
        });
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        if (n[t] >= N) continue;
#pragma unroll
        for (int a = 0; a < AG; ++a)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = 16 * (a0 + a) + 4 * g + i;
                if (m < M) out[(size_t)m * N + n[t]] = fs[a][t][i];
            }
    }
}

template <int MT, int NT, int U, int S>
mri_status launch_i8(const int8_t *act, size_t m, size_t kp, const float *sa_ptr,
                     int sa_stride, float sa_value, const QMatrixDev &w, float *out,
                     int32_t *acc_out, hipStream_t s) {
    constexpr int lds = S * MT * NT * 4 * kWave * 4;
    static_assert(lds <= 64 * 1024, "the waves' sums");
    hipLaunchKernelGGL((k_skinny_int8<MT, NT, U, S>), dim3((unsigned)((w.n_tiles + NT - 1) / NT)),
                       dim3(S * kWave), lds, s, act, (int)m, kp, sa_ptr, sa_stride,
                       sa_value, reinterpret_cast<const v4i *>(w.tiles), w.scales,
                       (int)w.n_out, (int)w.n_tiles, (int)(w.kp / kChunkK), out, acc_out);
    MRI_LAUNCHED("k_skinny_int8");
    return MRI_OK;
}
// Tiles and waves of a workgroup.  One tile while every CU has at most one
// workgroup, two up to two tiles a CU, then four: tiles that share a workgroup
// share its activation loads from L2, which bound the kernel, but 5 rows to 63
// fill a CU with one workgroup (us a call from f32, NT = 1 / 2 / 4: 32 x 5120 x
// 5120 25.4 / 17.8 / 21.1, 63 x 4096 x 8192 - / 21.0 / 24.3, 63 x 4096 x 11008
// - / 31.6 / 25.1; four from 512 tiles on, as before, 25.5 at 63 x 4096 x 8192).
// Waves: eight of two chunks in flight (32 x 11008 x 4096 23.8, sixteen 25.0;
// four tiles: four waves); for one tile of rows sixteen where K is 48 to 128
// chunks (5 x 4096 x 4096 9.4, eight 9.9) and four of four below (16 x 512 x
// 2048 7.0, 7.1).
template <int MT>
mri_status launch_i8_rows(const int8_t *act, size_t m, size_t kp, const float *sa_ptr,
                          int sa_stride, float sa_value, const QMatrixDev &w, float *out,
                          int32_t *acc_out, hipStream_t s) {
    const size_t chunks = w.kp / kChunkK, cus = (size_t)std::max(device_cus(), 1);
    if (w.n_tiles > 2 * cus)
        return launch_i8<MT, 4, 2, 4>(act, m, kp, sa_ptr, sa_stride, sa_value, w, out, acc_out, s);
    if (w.n_tiles > cus)
        return launch_i8<MT, 2, 2, 8>(act, m, kp, sa_ptr, sa_stride, sa_value, w, out, acc_out, s);
    if constexpr (MT == 1) {
        if (chunks < 48)
            return launch_i8<1, 1, 4, 4>(act, m, kp, sa_ptr, sa_stride, sa_value, w, out, acc_out, s);
        if (chunks < 128)
            return launch_i8<1, 1, 2, 16>(act, m, kp, sa_ptr, sa_stride, sa_value, w, out, acc_out, s);
    }
    return launch_i8<MT, 1, 2, 8>(act, m, kp, sa_ptr, sa_stride, sa_value, w, out, acc_out, s);
}

template <int I>
using Int = std::integral_constant<int, I>;

// AG activation groups per wave, ns waves per tile (AG * ns groups of 16 rows).
template <int AG, int NT, int RL, int CS, bool DEBUG, bool W4>
void launch_q8(const int8_t *act, size_t m, size_t kp, const float *sa_rows,
               const Q8MatrixDev &w, float *out, int32_t *block_dots, int ns, int mg,
               hipStream_t s) {
    const int G = (int)w.laps_per_tile();
    size_t grid = (w.n_tiles + NT - 1) / NT * (size_t)ns;
    if (ns > 1) grid = (grid + 7) / 8 * 8;  // XCD-major mapping (whole waves past the end exit)
    hipLaunchKernelGGL((k_skinny_q8_0<AG, NT, RL, CS, DEBUG, W4>),
                       dim3((unsigned)grid), dim3(kWave), 0, s,
                       act, (int)m, (int)kp, sa_rows, reinterpret_cast<const v4i *>(w.laps),
                       (int)w.n_out, (int)w.n_tiles, G,
                       (int)w.n_blocks, out, block_dots, ns, mg);
}

}  // namespace

mri_status launch_skinny_int8(const int8_t *act, size_t m, const float *sa_ptr,
                              int sa_stride, float sa_value,
                              const QMatrixDev &w, float *out,
                              int32_t *acc_out, hipStream_t s) {
    if (w.n_tiles == 0 || m == 0) return MRI_OK;
    const size_t kp = w.kp;
    for (size_t m0 = 0; m0 < m; m0 += 64) {
        const size_t mc = m - m0 < 64 ? m - m0 : 64;
        const int8_t *a = act + m0 * kp;
        const float *sp = sa_ptr ? sa_ptr + m0 * (size_t)sa_stride : nullptr;
        float *o = out + m0 * w.n_out;
        int32_t *ao = acc_out ? acc_out + m0 * w.n_out : nullptr;
        const mri_status st =
            mc <= 16   ? launch_i8_rows<1>(a, mc, kp, sp, sa_stride, sa_value, w, o, ao, s)
            : mc <= 32 ? launch_i8_rows<2>(a, mc, kp, sp, sa_stride, sa_value, w, o, ao, s)
                       : launch_i8_rows<4>(a, mc, kp, sp, sa_stride, sa_value, w, o, ao, s);
        if (st) return st;
    }
    return MRI_OK;
}

namespace {

// A wave takes AG groups of 16 rows of NT tiles; the waves of a tile are
// neighbouring workgroups of one XCD and share its weights in L2 (four of them
// in one workgroup: 2-10 % slower).  More groups a wave feed one weight
// operand to more MFMAs, more tiles one activation operand; fewer leave more
// waves, which 16 x 16 outputs a SIMD (u) decides.  us a call at K = 4096,
// AG x NT = 1 x 1 / 2 x 1 / 2 x 2 / 4 x 2, the best marked:
//   Q8_0    64 rows, 256 tiles (u = 1)    15.2* 19    -     -
//          128 rows, 256 tiles (u = 2)    22.4  19.5*  -     -
//           64 rows, 688 tiles (u = 2.7)   -    28.0* 28.8   -
//          100 rows, 688 tiles (u = 4.7)   -    41.4  38.8*  -
//           64 rows, 2000 tiles (u = 8)    -     -    49.8*  -
//          128 rows, 2000 tiles (u = 16)   -     -    84.7  74.1*
//         2048 rows, 688 tiles (u = 86)    -     -    418   357*
//   W4, whose weights cost half the bytes,
//           64 rows, 688 tiles (u = 2.7)  26.3* 26.9   -     -
//          127 rows, 688 tiles (u = 5.4)   -    38.1* 40.9   -
//          127 rows, 2000 tiles (u = 16)   -     -    85.3  79.1*
// Up to 16 rows, two tiles of Q8_0 from one wave a SIMD on (5 x 4096 x 22016
// 24.7 and 22.4).  Laps in flight of one group and tile: three, or two where K
// is eight laps or less (64 x 2048 x 4096 12.0 and 11.3) and W4 has several
// waves a SIMD (10 x 4096 x 20000 22.3 and 20.0).
// Before, with one tile a wave and one or two groups at every size, 2048 x 4096 x
// 11008 took 618 us and 127 x 4096 x 32000 111; now 368 and 77.
template <bool DEBUG>
void launch_q8_groups(const int8_t *act, size_t m, size_t kp, const float *sa_rows,
                      const Q8MatrixDev &w, float *out, int32_t *block_dots, int mg,
                      hipStream_t s) {
    auto go = [&](auto ag, auto nt, auto rl, auto cs) {
        constexpr int AG = decltype(ag)::value;
        const int ns = (int)((m + 16 * AG - 1) / (16 * AG));
        auto run = [&](auto w4) {
            launch_q8<AG, decltype(nt)::value, decltype(rl)::value, decltype(cs)::value, DEBUG,
                      decltype(w4)::value>(act, m, kp, sa_rows, w, out, block_dots, ns, mg, s);
        };
        constexpr bool q8_only = AG < decltype(nt)::value;
        if constexpr (!q8_only)
            if (w.w4) return run(std::true_type{});
        run(std::false_type{});
    };
    const Int<0> any{};
    const Int<1> one{};
    const Int<2> two{};
    const double u = (double)w.n_tiles * ((m + 15) / 16) / (4 * std::max(device_cus(), 1));
    if (m <= 16 && mg != 1) return go(one, one, two, Int<64>{});
    if constexpr (!DEBUG) {
        const bool laps2 = w.laps_per_tile() <= 8;
        if (m <= 16) {
            const Int<1024> group{};
            if (u > 1 && !w.w4) return go(one, two, two, group);
            if (u <= 1 && !laps2) return go(one, one, Int<3>{}, group);
            if (u <= 1024) return go(one, one, two, group);  // (2^30 channels: past the grid)
        }
        if (u <= (w.w4 ? 3 : 1))
            return laps2 ? go(one, one, two, any) : go(one, one, Int<3>{}, any);
        if (u > 12) return go(Int<4>{}, two, one, any);
        if (u > (w.w4 ? 6.5 : 3.5)) return go(two, two, two, any);
    }
    // (the block dots' registers leave room for no more)
    return u <= 1 ? go(one, one, two, any) : go(two, one, two, any);
}

}  // namespace

mri_status launch_skinny_q8_0(const int8_t *act, size_t m,
                              const float *sa_rows, const Q8MatrixDev &w,
                              float *out, int32_t *block_dots,
                              hipStream_t s, size_t mg) {
    if (w.n_tiles == 0 || m == 0) return MRI_OK;
    if (block_dots)
        launch_q8_groups<true>(act, m, w.kp, sa_rows, w, out, block_dots, (int)mg, s);
    else
        launch_q8_groups<false>(act, m, w.kp, sa_rows, w, out, nullptr, (int)mg, s);
    MRI_LAUNCHED("k_skinny_q8_0");
    return MRI_OK;
}

}  // namespace mri
