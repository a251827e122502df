// Device kernels of the MI355X (gfx950) batched ragged decode pass.
//
// Reference counterparts (l-wn/ChatTorrent, web/model/kernels.js) are cited
// per kernel. The design is MI355X-first: q8 projections run on MFMA
// (v_mfma_f32_16x16x32_f16) with the int8 codes dequantised exactly to f16 in
// registers and the f32 activations split into an f16 hi/lo pair, so each
// 32-wide quantisation group is one MFMA pair followed by one scale FMA per
// output; attention streams each chat's int8 pages once per kv head for the
// whole GQA group, also on MFMA; element-wise work is fused into the
// reduction ("finish") kernels that feed the next projection its operand.
#include "common.h"
#include "kernels.h"
#include <algorithm>
#include <mutex>
#include <type_traits>

// The first launch error since the last take_launch_error(); cc_step and the
// other entry points report it as CC_EDEVICE after their synchronisation.
static hipError_t g_launch_error = hipSuccess;
hipError_t take_launch_error() {
    hipError_t e = g_launch_error;
    g_launch_error = hipSuccess;
    return e;
}
#define CHECK_LAUNCH()                                                       \
    do {                                                                     \
        hipError_t e_ = hipGetLastError();                                   \
        if (e_ != hipSuccess && g_launch_error == hipSuccess) g_launch_error = e_; \
    } while (0)

// ===================================================================== GEMM ===
// Y[M, N] = X[M, K] . W[N, K]^T for a q8 W in record order (kernels.h) and an
// activation operand Xp prepared by the prep/finish kernels:
//   Xp[((mt*G2 + g)*2 + hl)*64 + lane] = 8 f16 of X[16mt + lane%16][32g + 8(lane/16) ..]
// (hl = 0: hi part, 1: lo part scaled by 2^11 (split_hilo_x), which meets the
// weights scaled by 2^-11; G2 = 2*KU groups, zero beyond K).
// Reference: matmul_gemv_q8 / matmul_gemv_rows_q8 / matmul_rows_q8 /
// matmul_tiled_q8 (web/model/kernels.js:449-804): per group, acc += scale * dot(x, q).
//
// Workgroup g (8 waves) serves plane r = g % P and a contiguous block of tile
// pairs; it first copies the plane's activations (MT m-tiles x <= LX_UNITS
// units, <= 160 KiB) into LDS, so the waves' only global loads are the weight
// records, which stream LX_R - 1 steps ahead. A "step" is one (pair, unit)
// record; the workgroup's steps are split evenly over its waves in record
// order, so each wave reads one forward run of memory. A pair cut between
// waves is finished by the wave holding its first units, adding the others'
// parts in unit order; the parts meet in LDS once every wave is past its last
// step (the activations are dead by then). Every split point depends on N, K
// and the CU count, never on M, so a row's result is the same in any batch.
// Output: plane r to out[(r*M + m)*N + n]; consumers add planes 0..P-1 in order
// (gemm_planes: one plane when k_gemm_tm_sum has added them).
constexpr int LX_WAVES = 8;
// The weight ring: one record in flight a wave ahead of the one computed.
// Measured at configs[2]: two or three records ahead made the pass 4-6%
// slower (more requests outstanding across the GPU's 2048 waves), none ahead
// 13% slower.
constexpr int LX_R = 2;

typedef __attribute__((address_space(3))) void lds_void_t;

// The scale of half-group h (K columns 32h .. 32h+31 of the unit) of one
// tile row, from the row's 32-bit word in the record's scale block: an f16
// per 32-wide group (h = 0 in the low half), or one f32 per 64-wide unit
// that both halves share (QTensor::f32s).
template <bool F32S>
__device__ static inline float rec_scale(uint32_t word, int h) {
    if constexpr (F32S) {
        (void)h;
        return __builtin_bit_cast(float, word);
    } else {
        const uint16_t s16 = h ? (uint16_t)(word >> 16) : (uint16_t)(word & 0xffffu);
        return (float)__builtin_bit_cast(_Float16, s16);
    }
}

// Few rows (launch_gemm_resid, launch_gemm_swiglu; gemm_fuses says when): the workgroup forms its
// plane's operand itself from the previous projection's planes, in place of
// k_resid_w's or k_fin_swiglu's launch and the operand's way through memory:
// the same values by the same operations, in as many places as there are
// column groups. LX_PRO_RESID's grid has workgroups after the matmul's, four
// (512-column slice, row) pairs each, that store the new residual rows (in
// another buffer: the others still read the old ones) and the sums of squares.
// The operand's rows past M stay whatever LDS held: a row of the product
// depends on its own row alone, and rows past M are not stored.
// LX_PRO_ATTN does the same with k_attn_combine's launch (gemm_fuses_attn).
// Few rows leave each launch bound by its own start, drain and first loads:
// three of a block's ten go, or four. One chat: hidden 576, 30 blocks and
// head 1254 -> 1083 us, and with attention's merge, after four waves an
// attention item, 1045 -> 977; hidden 5120, 4 blocks 502 -> 470 us.
__device__ static inline float row_scale(const RowScale& rs, int m);
constexpr int LX_PRO_NONE = 0, LX_PRO_RESID = 1, LX_PRO_SWIGLU = 2, LX_PRO_ATTN = 3;
struct LxPro {
    const float* part = nullptr;   // the previous projection's planes (ATTN: the chunk partials)
    int splits = 0;
    const float* x = nullptr;      // RESID: residual rows, the new ones, the norm's weights
    float* xo = nullptr;
    const float* w = nullptr;
    int round = 0;
    float* ssp = nullptr;
    int G = 0;                     // the matmul's workgroups
    RowScale rs;                   // SWIGLU: the row factor
    int F = 0;
    const JobDev* jobs = nullptr;  // ATTN: the rows' jobs, the output gate or null, head_dim, query heads a KV head
    const int32_t* row_job = nullptr;
    const float* gate = nullptr;
    int D = 0, group = 0;
};
struct LxNoPro {};
template <int PRO>
struct LxProArg { using type = LxPro; };
template <>
struct LxProArg<LX_PRO_NONE> { using type = LxNoPro; };   // no prologue, no arguments of one
template <int N>
__device__ static inline void resid_row(const LxPro& p, int M, int H, int m, int k0, float (&x)[N]);
__device__ static inline void swiglu8(const LxPro& p, int M, int m, int k0, float f, float (&v)[8]);
__device__ static void resid_slices(const LxPro& p, int M, int H, float* red);
__device__ static inline void combine4(const LxPro& p, int K, int m, int unit, int lane, float (&v)[4]);

template <int MT, bool F32S, int PRO = LX_PRO_NONE>
__global__ __launch_bounds__(64 * LX_WAVES) void k_gemm_lx(const uint8_t* __restrict__ Wr,
                                                           const uint4* __restrict__ Xp, float* __restrict__ out,
                                                           int KU, int M, int N, int Nt, int P, int Gm,
                                                           typename LxProArg<PRO>::type pro) {
    static_assert(PRO == LX_PRO_NONE || MT == 1, "a prologue forms one m-tile");
    constexpr int NT = 2, R = LX_R, PW = R - 1, WAVES = LX_WAVES;
    extern __shared__ __attribute__((aligned(1024))) u32x4 xs[];
    if constexpr (PRO == LX_PRO_RESID)
        if ((int)blockIdx.x >= pro.G) {
            resid_slices(pro, M, 64 * KU, (float*)xs);
            return;
        }
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = blockIdx.x % P, j = blockIdx.x / P;
    const int ua = lx_plane_start(r, KU, P), len = lx_plane_start(r + 1, KU, P) - ua;
    const int npairs = Nt / NT;
    const int p0 = (j * npairs) / Gm, p1 = ((j + 1) * npairs) / Gm;
    const int steps = (p1 - p0) * len;
    const int sw0 = (wave * steps) / WAVES, sw1 = ((wave + 1) * steps) / WAVES;
    const int nst = sw1 - sw0;
    const int mt0 = blockIdx.y * MT;
    const int G2 = 2 * KU;
    const auto rw = __builtin_amdgcn_make_buffer_rsrc((void*)Wr, 0, 0x7fffffff, 0x00020000);
    const auto rx = __builtin_amdgcn_make_buffer_rsrc((void*)Xp, 0, 0x7fffffff, 0x00020000);
    // Plane r's rows only: stores of rows >= M fall outside and are dropped.
    const auto ro = __builtin_amdgcn_make_buffer_rsrc((void*)(out + (size_t)r * M * N), 0, M * N * 4, 0x00020000);
    const int vw = lane * 16, vs = NT * 1024 + (lane & 15) * NT * 4;
    const int vo = (4 * (lane >> 4) * N + (lane & 15)) * 4;
    const int rec0 = ua * npairs + p0 * len;

    u32x4 w[R][NT];
    uint32_t s[R][NT];
    int sl = sw0;   // next step to load; stays on the last one past the end
    auto load_w = [&](u32x4 (&wv)[NT], uint32_t (&sv)[NT]) {
        const int off = (rec0 + sl) * LX_REC;
        wv[0] = __builtin_amdgcn_raw_buffer_load_b128(rw, vw, off, 2);
        wv[1] = __builtin_amdgcn_raw_buffer_load_b128(rw, vw, off + 1024, 2);
        const auto sc = __builtin_amdgcn_raw_buffer_load_b64(rw, vs, off, 0);
        sv[0] = sc[0];
        sv[1] = sc[1];
        if (sl + 1 < sw1) sl++;
    };
    if (nst > 0) {
#pragma unroll
        for (int i = 0; i < PW; i++) load_w(w[i], s[i]);
    }
    // Activations of this plane into LDS: block (u, mt, q) of 1 KiB, q = 2h + hl.
    if constexpr (PRO == LX_PRO_ATTN) {
        // a wave's 64 columns of a row at a time
        for (int i = wave; i < M * len; i += WAVES) {
            const int m = i / len, u = i % len;
            float v[4];
            combine4(pro, 64 * KU, m, ua + u, lane, v);
            if (lane < 16) {
                _Float16 h[4], l[4];
#pragma unroll
                for (int e = 0; e < 4; e++) split_hilo_x(v[e], h[e], l[e]);
                // columns 4 lane ..: half-group lane / 8, k-block (lane % 8) / 2, half of its 16 bytes
                uint2* at = (uint2*)(xs + (u * 4 + 2 * (lane >> 3)) * 64 + m + 16 * ((lane & 7) >> 1)) + (lane & 1);
                at[0] = make_uint2(__builtin_bit_cast(uint32_t, half2_t{h[0], h[1]}),
                                   __builtin_bit_cast(uint32_t, half2_t{h[2], h[3]}));
                at[128] = make_uint2(__builtin_bit_cast(uint32_t, half2_t{l[0], l[1]}),
                                     __builtin_bit_cast(uint32_t, half2_t{l[2], l[3]}));
            }
        }
    } else if constexpr (PRO != LX_PRO_NONE) {
        // a thread's 8 columns of a row at a time
        const int per = 8 * len;
        for (int i = threadIdx.x; i < M * per; i += 64 * WAVES) {
            const int m = i / per, c = i % per, k0 = 64 * ua + 8 * c;
            float v[8];
            if constexpr (PRO == LX_PRO_RESID) {
                resid_row<8>(pro, M, 64 * KU, m, k0, v);
                const float4 wa = *(const float4*)(pro.w + k0), wb = *(const float4*)(pro.w + k0 + 4);
                const float wv[8] = {wa.x, wa.y, wa.z, wa.w, wb.x, wb.y, wb.z, wb.w};
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = v[e] * wv[e];
            } else
                swiglu8(pro, M, m, k0, row_scale(pro.rs, m), v);
            half8_t hi, lo;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                _Float16 a, b;
                split_hilo_x(v[e], a, b);
                hi[e] = a;
                lo[e] = b;
            }
            // unit c / 8, half-group (c % 8) / 4, k-block c % 4
            u32x4* at = xs + ((c >> 3) * 4 + 2 * ((c >> 2) & 1)) * 64 + m + 16 * (c & 3);
            at[0] = __builtin_bit_cast(u32x4, hi);
            at[64] = __builtin_bit_cast(u32x4, lo);
        }
    } else {
        const int nblk = len * MT * 4;
        for (int b = wave; b < nblk; b += WAVES) {
            const int u = b / (MT * 4), mt = (b / 4) % MT, q = b % 4;
            const int src = ((mt0 + mt) * G2 + 2 * (ua + u) + (q >> 1)) * 2 + (q & 1);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void_t*)(xs + b * 64), 16, vw, src * 1024, 0, 0);
        }
    }
    float4_t acc[MT][NT], tail[MT][NT];   // tail: this wave's part of a pair begun in an earlier wave
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) acc[mt][nt] = tail[mt][nt] = float4_t{0.f, 0.f, 0.f, 0.f};
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();

    auto compute = [&](const u32x4 (&wc)[NT], const uint32_t (&sc)[NT], int u) {
        u32x4 xv[MT][4];
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int q = 0; q < 4; q++) xv[mt][q] = xs[((u * MT + mt) * 4 + q) * 64 + lane];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            half8_t b[NT];
            float scale[NT];
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                b[nt] = h ? dequant8_biased(wc[nt][2], wc[nt][3]) : dequant8_biased(wc[nt][0], wc[nt][1]);
                scale[nt] = rec_scale<F32S>(sc[nt], h);
            }
            // hi then lo into one partial per output, then one scale FMA
            float4_t pp[MT][NT];
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
                    pp[mt][nt] = mfma16x16x32(__builtin_bit_cast(half8_t, xv[mt][2 * h]), b[nt],
                                              float4_t{0.f, 0.f, 0.f, 0.f});
            half8_t bl[NT];   // the lo half carries 2^11 x its remainder
#pragma unroll
            for (int nt = 0; nt < NT; nt++) bl[nt] = lo_weight8(b[nt]);
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
                    pp[mt][nt] = mfma16x16x32(__builtin_bit_cast(half8_t, xv[mt][2 * h + 1]), bl[nt], pp[mt][nt]);
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        acc[mt][nt][e] = __builtin_fmaf(scale[nt], pp[mt][nt][e], acc[mt][nt][e]);
        }
    };
    auto store_plane = [&](int pair) {
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            const int tile = (p0 + pair) * NT + nt;
            if (tile * 16 >= N) continue;
            // columns past N of a partial tile would land in the next row
            if (tile * 16 + 16 > N && tile * 16 + (lane & 15) >= N) continue;
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float v = acc[mt][nt][e];
                    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), ro,
                                                          vo + (((mt0 + mt) * 16 + e) * N + tile * 16) * 4, 0, 0);
                }
        }
    };
    int pc = 0, uc = 0;   // (pair, unit) of the step being computed
    if (nst > 0) {
        pc = sw0 / len;
        uc = sw0 - pc * len;
    }
    bool head_open = false, has_tail = false;
    // After a pair's last unit (or this wave's last step) its partial goes to
    // `out` (whole pair), to `tail` (pair began in an earlier wave), or stays
    // in acc (pair goes on in later waves).
    auto finish_step = [&](int st) {
        if (uc == len - 1 || st == sw1 - 1) {
            if (pc * len < sw0) {
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
#pragma unroll
                    for (int nt = 0; nt < NT; nt++) tail[mt][nt] = acc[mt][nt];
                has_tail = true;
            } else if ((pc + 1) * len <= sw1) {
                store_plane(pc);
            } else {
                head_open = true;
            }
            if (!head_open) {
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
#pragma unroll
                    for (int nt = 0; nt < NT; nt++) acc[mt][nt] = float4_t{0.f, 0.f, 0.f, 0.f};
            }
        }
        if (++uc == len) {
            uc = 0;
            pc++;
        }
    };
    if (nst > 0) {
        int k = 0;
        for (; k + R <= nst; k += R) {
#pragma unroll
            for (int I = 0; I < R; I++) {
                load_w(w[(I + PW) % R], s[(I + PW) % R]);
                __builtin_amdgcn_sched_barrier(0);
                compute(w[I], s[I], uc);
                __builtin_amdgcn_sched_barrier(0);
                finish_step(sw0 + k + I);
            }
        }
        // At most PW steps remain, already in ring slots 0 .. PW-1.
#pragma unroll
        for (int I = 0; I < PW; I++) {
            if (k + I < nst) {
                compute(w[I], s[I], uc);
                finish_step(sw0 + k + I);
            }
        }
    }
    // Every wave is past its last step: the LDS activations are dead and hold
    // the cut parts now, one 1 KiB slot per (wave, m-tile, tile).
    __syncthreads();
    if (has_tail) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++)
                xs[((wave * MT + mt) * NT + nt) * 64 + lane] = __builtin_bit_cast(u32x4, tail[mt][nt]);
    }
    __syncthreads();
    if (head_open) {
        const int pair = (sw1 - 1) / len, pe = (pair + 1) * len;
        for (int w2 = wave + 1; w2 < WAVES; w2++) {
            const int a2 = (w2 * steps) / WAVES, b2 = ((w2 + 1) * steps) / WAVES;
            if (a2 >= pe) break;
            if (b2 <= a2) continue;
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++) {
                    const float4_t o = __builtin_bit_cast(float4_t, xs[((w2 * MT + mt) * NT + nt) * 64 + lane]);
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[mt][nt][e] = acc[mt][nt][e] + o[e];
                }
        }
        store_plane(pair);
    }
}

int lx_groups(const QTensor& w, int ncu) {
    const int per = std::max(1, std::min(ncu / w.P, w.Nt / 2));
    return w.P * per;
}

// K planes of an N x K q8 tensor: the fewest the LDS allows (lx_planes),
// doubled (up to 16, and to one unit a plane) while the workgroups the
// matmul launches (planes x column groups, lx_groups) would fill fewer than
// half the CUs. A small model's narrow matrices (30 tile pairs at
// SmolLM2's q|k|v) otherwise leave most CUs idle; a 27B or 8B layer fills
// them at the fewest planes and keeps those.
int lx_planes_for(int N, int K, int ncu) {
    const int KU = (K + 63) / 64, npairs = (N + 31) / 32;
    int P = lx_planes(KU);
    while (2 * P <= std::min(KU, 16) && 2LL * P * std::max(1, std::min(ncu / P, npairs)) <= ncu) P *= 2;
    return P;
}

template <int MT, bool F32S, int PRO = LX_PRO_NONE>
static void launch_lx(hipStream_t st, const QTensor& w, const uint4* Xp, float* out, int M, int ncu,
                      typename LxProArg<PRO>::type pro = {}) {
    static bool attr = false;
    if (!attr) {
        attr = true;
        (void)hipFuncSetAttribute((const void*)k_gemm_lx<MT, F32S, PRO>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  LX_UNITS * MT * 4096);
    }
    const int G = lx_groups(w, ncu), Gm = G / w.P;
    const int lenmax = (w.KU + w.P - 1) / w.P;
    // the plane's activations, and afterwards the cut parts (1 KiB per wave, m-tile and tile)
    const size_t lds = std::max((size_t)lenmax * MT * 4096, (size_t)LX_WAVES * MT * 2 * 1024);
    if constexpr (PRO != LX_PRO_NONE) pro.G = G;
    const int extra = PRO == LX_PRO_RESID ? (M * ((w.K / 4 + RW_THREADS - 1) / RW_THREADS) + 3) / 4 : 0;
    dim3 grid(G + extra, (M + 16 * MT - 1) / (16 * MT));
    hipLaunchKernelGGL((k_gemm_lx<MT, F32S, PRO>), grid, dim3(64 * LX_WAVES), lds, st, (const uint8_t*)w.codes, Xp,
                       out, w.KU, M, w.N, w.Nt, w.P, Gm, pro);
}

// ------------------------------------------------- many rows (M > 32) ---
// Above 32 rows k_gemm_lx would stream every weight once per 32-row block.
// k_gemm_tm reuses each weight record across 64 rows instead: a workgroup
// serves plane r (the same planes as k_gemm_lx), TM_PAIRS tile pairs and 64
// rows (4 m-tiles); wave (h, i) computes rows 32h .. 32h+31 of pair i, so
// each record feeds two waves. The activations of one unit of K for the 64
// rows (16 KiB) are staged through registers into a double-buffered LDS
// block, one barrier a unit, while each wave streams its pair's records
// TM_R-1 units ahead (144 VGPRs: two waves a SIMD).
//
// Bits: a row's result is bit-identical to k_gemm_lx's at any M. Within a
// plane k_gemm_lx sums a pair's units in order but in segments, cut where
// its workgroup's steps are split between waves, and adds the segments in
// order; the cut points depend only on N, K and the CU count (lx_cuts), and
// k_gemm_tm folds its running sum at the same units. Each MFMA pair, scale
// FMA and addition is the same operation on the same operands.
constexpr int TM_MT = 4, TM_WAVES = 8, TM_PAIRS = 8, TM_R = 2;

// Unit offsets inside pair p (of a plane of `len` <= 32 units) where
// k_gemm_lx starts a new partial sum, as a bit mask: the wave boundaries of
// the lx workgroup holding p (workgroup j of Gm covers pairs
// [j*npairs/Gm, (j+1)*npairs/Gm)) that fall strictly inside the pair.
__device__ static inline uint32_t lx_cuts(int p, int npairs, int Gm, int len) {
    // In closed form with 32-bit divisions (npairs * Gm < 2^31: a weight is
    // under 2 GB, and Gm at most the CU count). A search with 64-bit divisions
    // took about 700 scalar instructions, 1-2 us of every many-row workgroup's
    // 25: gate|up at 1088 rows 931 -> 888 us (27B) and 633 -> 611 (8B).
    const uint32_t np = (uint32_t)npairs, g = (uint32_t)Gm;
    const uint32_t j = (((uint32_t)p + 1) * g - 1) / np;   // the last j with floor(j*np/g) <= p
    const int p0 = (int)(j * np / g), p1 = (int)((j + 1) * np / g);
    const int steps = (p1 - p0) * len, s0 = (p - p0) * len;
    uint32_t m = 0;
#pragma unroll
    for (int w = 1; w < LX_WAVES; w++) {
        const int b = (w * steps) / LX_WAVES - s0;
        if (b > 0 && b < len) m |= 1u << b;
    }
    return m;
}

template <bool F32S>
__global__ __launch_bounds__(64 * TM_WAVES) void k_gemm_tm(const uint8_t* __restrict__ Wr,
                                                              const uint4* __restrict__ Xp, int xp_mtiles,
                                                              float* __restrict__ out, int KU, int M, int N, int Nt,
                                                              int P, int Gm) {
    constexpr int NT = 2, R = TM_R, PW = R - 1, MTL = TM_MT, MTW = MTL * TM_PAIRS / TM_WAVES;
    static_assert(MTW * TM_WAVES == MTL * TM_PAIRS, "waves cover pairs x m-tiles");
    __shared__ u32x4 xs[2][MTL * 4][64];   // two units: block (m-tile, q = 2h + hl) of 1 KiB
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int npairs = Nt / NT;
    // Workgroups b and b + 8 run on one XCD (dispatch is round-robin over the
    // XCDs, from an offset that varies by launch).
    // Each (plane, pair group) goes to one XCD, which runs its row blocks back
    // to back, so the row blocks after the first read its weight records from
    // that XCD's L2 instead of HBM. The order of workgroups changes no sums.
    const int nrb = (M + 16 * MTL - 1) / (16 * MTL), npg = (npairs + TM_PAIRS - 1) / TM_PAIRS;
    const int kx = blockIdx.x / 8;
    const int gx = (kx / nrb) * 8 + blockIdx.x % 8, gy = kx % nrb;
    if (gx >= P * npg) return;   // the grid is rounded up to whole XCD rounds
    const int r = gx % P, pb = gx / P;
    const int pair = pb * TM_PAIRS + wave % TM_PAIRS, mw = (wave / TM_PAIRS) * MTW;   // m-tiles mw .. mw+MTW-1
    const bool has = pair < npairs;
    const int ua = lx_plane_start(r, KU, P), len = lx_plane_start(r + 1, KU, P) - ua;
    const int mt0 = gy * MTL;
    const int G2 = 2 * KU;
    const auto rw = __builtin_amdgcn_make_buffer_rsrc((void*)Wr, 0, 0x7fffffff, 0x00020000);
    // activation m-tiles past the operand's allocation read zero
    const uint32_t xbytes = (uint32_t)min((unsigned long long)xp_mtiles * G2 * 2048ull, 0xffffffffull);
    const auto rx = __builtin_amdgcn_make_buffer_rsrc((void*)Xp, 0, xbytes, 0x00020000);
    const auto ro = __builtin_amdgcn_make_buffer_rsrc((void*)(out + (size_t)r * M * N), 0, M * N * 4, 0x00020000);
    const int vw = lane * 16, vs = NT * 1024 + (lane & 15) * NT * 4;
    const int vo = (4 * (lane >> 4) * N + (lane & 15)) * 4;
    const int rec0 = (ua * npairs + (has ? pair : 0) * len) * LX_REC;
    const uint32_t cuts = has ? lx_cuts(pair, npairs, Gm, len) : 0u;

    // this wave's share of a unit's activations: blocks BPW*wave .. +BPW-1
    constexpr int BPW = MTL * 4 / TM_WAVES;
    static_assert(BPW * TM_WAVES == MTL * 4, "activation blocks split evenly over the waves");
    u32x4 st[BPW];
    auto load_x = [&](int u) {
        const int Uk = ua + (u < len ? u : len - 1);
#pragma unroll
        for (int k = 0; k < BPW; k++) {
            const int b = BPW * wave + k, mt = b >> 2, q = b & 3;
            const int src = ((mt0 + mt) * G2 + 2 * Uk + (q >> 1)) * 2 + (q & 1);
            st[k] = __builtin_amdgcn_raw_buffer_load_b128(rx, vw, src * 1024, 0);
        }
    };
    auto store_x = [&](int buf) {
#pragma unroll
        for (int k = 0; k < BPW; k++) xs[buf][BPW * wave + k][lane] = st[k];
    };
    u32x4 w[R][NT];
    uint32_t sc[R][NT];
    auto load_w = [&](int u, u32x4 (&wv)[NT], uint32_t (&sv)[NT]) {
        const int off = rec0 + (u < len ? u : len - 1) * LX_REC;
        wv[0] = __builtin_amdgcn_raw_buffer_load_b128(rw, vw, off, 2);
        wv[1] = __builtin_amdgcn_raw_buffer_load_b128(rw, vw, off + 1024, 2);
        const auto s2 = __builtin_amdgcn_raw_buffer_load_b64(rw, vs, off, 0);
        sv[0] = s2[0];
        sv[1] = s2[1];
    };
    float4_t seg[MTW][NT], tot[MTW][NT];
#pragma unroll
    for (int mt = 0; mt < MTW; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) seg[mt][nt] = tot[mt][nt] = float4_t{0.f, 0.f, 0.f, 0.f};
    bool started = false;   // tot holds the first segment(s)

    load_x(0);
#pragma unroll
    for (int i = 0; i < PW; i++) load_w(i, w[i], sc[i]);
    store_x(0);
    load_x(1);
    __syncthreads();

    auto unit = [&](int u, const u32x4 (&wc)[NT], const uint32_t (&sv)[NT]) {
        const int buf = u & 1;
        // the unit k_gemm_lx begins a new partial sum at: fold the running one
        if ((cuts >> u) & 1u) {
#pragma unroll
            for (int mt = 0; mt < MTW; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++) {
                    if (started)
#pragma unroll
                        for (int e = 0; e < 4; e++) tot[mt][nt][e] = tot[mt][nt][e] + seg[mt][nt][e];
                    else
                        tot[mt][nt] = seg[mt][nt];
                    seg[mt][nt] = float4_t{0.f, 0.f, 0.f, 0.f};
                }
            started = true;
        }
        half8_t b[2][NT], bl[2][NT];   // bl: the lo half's fragment, 2^-11 b
        float scale[2][NT];
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                b[h][nt] = h ? dequant8_biased(wc[nt][2], wc[nt][3]) : dequant8_biased(wc[nt][0], wc[nt][1]);
                bl[h][nt] = lo_weight8(b[h][nt]);
                scale[h][nt] = rec_scale<F32S>(sv[nt], h);
            }
        // per half-group, every m-tile's MFMA pair first and the scale FMAs
        // after them, so no FMA waits on the MFMA issued just before it; each
        // output's operations and their order are those of k_gemm_lx
#pragma unroll
        for (int h = 0; h < 2; h++) {
            u32x4 xv[MTW][2];
#pragma unroll
            for (int mt = 0; mt < MTW; mt++)
#pragma unroll
                for (int q = 0; q < 2; q++) xv[mt][q] = xs[buf][(mw + mt) * 4 + 2 * h + q][lane];
            float4_t pp[MTW][NT];
#pragma unroll
            for (int mt = 0; mt < MTW; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
                    pp[mt][nt] = mfma16x16x32(__builtin_bit_cast(half8_t, xv[mt][0]), b[h][nt], float4_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int mt = 0; mt < MTW; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
                    pp[mt][nt] = mfma16x16x32(__builtin_bit_cast(half8_t, xv[mt][1]), bl[h][nt], pp[mt][nt]);
#pragma unroll
            for (int mt = 0; mt < MTW; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
#pragma unroll
                    for (int e = 0; e < 4; e++) seg[mt][nt][e] = __builtin_fmaf(scale[h][nt], pp[mt][nt][e], seg[mt][nt][e]);
        }
    };
    int u = 0;
    for (; u + R <= len; u += R) {
#pragma unroll
        for (int I = 0; I < R; I++) {
            load_w(u + I + PW, w[(I + PW) % R], sc[(I + PW) % R]);
            unit(u + I, w[I], sc[I]);
            // the next unit's activations go in the other buffer: every wave
            // finished reading it (one unit ago) before the last barrier
            store_x((I + 1) & 1);
            load_x(u + I + 2);
            __syncthreads();
        }
    }
    // at most PW units remain, their records in ring slots 0 .. PW-1
#pragma unroll
    for (int I = 0; I < PW; I++) {
        if (u + I < len) {
            unit(u + I, w[I], sc[I]);
            store_x((I + 1) & 1);
            load_x(u + I + 2);
            __syncthreads();
        }
    }
    if (!has) return;
#pragma unroll
    for (int mt = 0; mt < MTW; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            if (started)
#pragma unroll
                for (int e = 0; e < 4; e++) tot[mt][nt][e] = tot[mt][nt][e] + seg[mt][nt][e];
            else
                tot[mt][nt] = seg[mt][nt];
        }
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        const int tile = pair * NT + nt;
        if (tile * 16 >= N) continue;
        if (tile * 16 + 16 > N && tile * 16 + (lane & 15) >= N) continue;
#pragma unroll
        for (int mt = 0; mt < MTW; mt++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(tot[mt][nt][e]), ro,
                                                      vo + (((mt0 + mw + mt) * 16 + e) * N + tile * 16) * 4, 0, 0);
    }
}

// k_gemm_tm12: k_gemm_tm at twelve waves a workgroup (three a SIMD), each
// still one tile pair over the row block's 4 m-tiles, for matrices whose
// pair groups of twelve still give every CU a workgroup. The running sum of
// the segments already folded (k_gemm_tm's `tot`) lives in the wave's own
// LDS slot (8 KiB a wave) instead of 32 registers, which brings the kernel
// to 160 VGPRs: three waves a SIMD. A fold reads the slot, adds the segment
// and writes it back: the same additions in the same order, so every output
// keeps k_gemm_tm's (and k_gemm_lx's) bits. The staged activation blocks of
// a unit (16) are shared out over the twelve waves, one or two each.
constexpr int TM12_WAVES = 12;
template <bool F32S>
__global__ __launch_bounds__(64 * TM12_WAVES) void k_gemm_tm12(const uint8_t* __restrict__ Wr,
                                                              const uint4* __restrict__ Xp, int xp_mtiles,
                                                              float* __restrict__ out, int KU, int M, int N, int Nt,
                                                              int P, int Gm) {
    constexpr int NT = 2, R = TM_R, PW = R - 1, MTL = TM_MT, WV = TM12_WAVES;
    __shared__ u32x4 xs[2][MTL * 4][64];
    __shared__ float4_t tl[WV][MTL * NT][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int npairs = Nt / NT;
    const int nrb = (M + 16 * MTL - 1) / (16 * MTL), npg = (npairs + WV - 1) / WV;
    const int kx = blockIdx.x / 8;
    const int gx = (kx / nrb) * 8 + blockIdx.x % 8, gy = kx % nrb;
    if (gx >= P * npg) return;
    const int r = gx % P, pb = gx / P;
    const int pair = pb * WV + wave;
    const bool has = pair < npairs;
    const int ua = lx_plane_start(r, KU, P), len = lx_plane_start(r + 1, KU, P) - ua;
    const int mt0 = gy * MTL;
    const int G2 = 2 * KU;
    const auto rw = __builtin_amdgcn_make_buffer_rsrc((void*)Wr, 0, 0x7fffffff, 0x00020000);
    const uint32_t xbytes = (uint32_t)min((unsigned long long)xp_mtiles * G2 * 2048ull, 0xffffffffull);
    const auto rx = __builtin_amdgcn_make_buffer_rsrc((void*)Xp, 0, xbytes, 0x00020000);
    const auto ro = __builtin_amdgcn_make_buffer_rsrc((void*)(out + (size_t)r * M * N), 0, M * N * 4, 0x00020000);
    const int vw = lane * 16, vs = NT * 1024 + (lane & 15) * NT * 4;
    const int vo = (4 * (lane >> 4) * N + (lane & 15)) * 4;
    const int rec0 = (ua * npairs + (has ? pair : 0) * len) * LX_REC;
    const uint32_t cuts = has ? lx_cuts(pair, npairs, Gm, len) : 0u;
    constexpr int NB = MTL * 4, BPW = (NB + WV - 1) / WV;
    u32x4 st[BPW];
    auto load_x = [&](int u) {
        const int Uk = ua + (u < len ? u : len - 1);
#pragma unroll
        for (int k = 0; k < BPW; k++) {
            const int b = wave + k * WV, mt = b >> 2, q = b & 3;
            if (b < NB) {
                const int src = ((mt0 + mt) * G2 + 2 * Uk + (q >> 1)) * 2 + (q & 1);
                st[k] = __builtin_amdgcn_raw_buffer_load_b128(rx, vw, src * 1024, 0);
            }
        }
    };
    auto store_x = [&](int buf) {
#pragma unroll
        for (int k = 0; k < BPW; k++) {
            const int b = wave + k * WV;
            if (b < NB) xs[buf][b][lane] = st[k];
        }
    };
    u32x4 w[R][NT];
    uint32_t sc[R][NT];
    auto load_w = [&](int u, u32x4 (&wv)[NT], uint32_t (&sv)[NT]) {
        const int off = rec0 + (u < len ? u : len - 1) * LX_REC;
        wv[0] = __builtin_amdgcn_raw_buffer_load_b128(rw, vw, off, 2);
        wv[1] = __builtin_amdgcn_raw_buffer_load_b128(rw, vw, off + 1024, 2);
        const auto s2 = __builtin_amdgcn_raw_buffer_load_b64(rw, vs, off, 0);
        sv[0] = s2[0];
        sv[1] = s2[1];
    };
    float4_t seg[MTL][NT];
#pragma unroll
    for (int mt = 0; mt < MTL; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) seg[mt][nt] = float4_t{0.f, 0.f, 0.f, 0.f};
    bool started = false;

    load_x(0);
#pragma unroll
    for (int i = 0; i < PW; i++) load_w(i, w[i], sc[i]);
    store_x(0);
    load_x(1);
    __syncthreads();

    auto fold = [&]() {
#pragma unroll
        for (int mt = 0; mt < MTL; mt++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                float4_t t = seg[mt][nt];
                if (started) {
                    const float4_t o = tl[wave][mt * NT + nt][lane];
#pragma unroll
                    for (int e = 0; e < 4; e++) t[e] = o[e] + seg[mt][nt][e];
                }
                tl[wave][mt * NT + nt][lane] = t;
                seg[mt][nt] = float4_t{0.f, 0.f, 0.f, 0.f};
            }
        started = true;
    };
    auto unit = [&](int u, const u32x4 (&wc)[NT], const uint32_t (&sv)[NT]) {
        const int buf = u & 1;
        if ((cuts >> u) & 1u) fold();
        half8_t b[2][NT], bl[2][NT];
        float scale[2][NT];
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                b[h][nt] = h ? dequant8_biased(wc[nt][2], wc[nt][3]) : dequant8_biased(wc[nt][0], wc[nt][1]);
                bl[h][nt] = lo_weight8(b[h][nt]);
                scale[h][nt] = rec_scale<F32S>(sv[nt], h);
            }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            u32x4 xv[MTL][2];
#pragma unroll
            for (int mt = 0; mt < MTL; mt++)
#pragma unroll
                for (int q = 0; q < 2; q++) xv[mt][q] = xs[buf][mt * 4 + 2 * h + q][lane];
            float4_t pp[MTL][NT];
#pragma unroll
            for (int mt = 0; mt < MTL; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
                    pp[mt][nt] = mfma16x16x32(__builtin_bit_cast(half8_t, xv[mt][0]), b[h][nt], float4_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int mt = 0; mt < MTL; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
                    pp[mt][nt] = mfma16x16x32(__builtin_bit_cast(half8_t, xv[mt][1]), bl[h][nt], pp[mt][nt]);
#pragma unroll
            for (int mt = 0; mt < MTL; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
#pragma unroll
                    for (int e = 0; e < 4; e++) seg[mt][nt][e] = __builtin_fmaf(scale[h][nt], pp[mt][nt][e], seg[mt][nt][e]);
        }
    };
    int u = 0;
    for (; u + R <= len; u += R) {
#pragma unroll
        for (int I = 0; I < R; I++) {
            load_w(u + I + PW, w[(I + PW) % R], sc[(I + PW) % R]);
            unit(u + I, w[I], sc[I]);
            store_x((I + 1) & 1);
            load_x(u + I + 2);
            __syncthreads();
        }
    }
#pragma unroll
    for (int I = 0; I < PW; I++) {
        if (u + I < len) {
            unit(u + I, w[I], sc[I]);
            store_x((I + 1) & 1);
            load_x(u + I + 2);
            __syncthreads();
        }
    }
    if (!has) return;
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        const int tile = pair * NT + nt;
        if (tile * 16 >= N) continue;
        if (tile * 16 + 16 > N && tile * 16 + (lane & 15) >= N) continue;
#pragma unroll
        for (int mt = 0; mt < MTL; mt++) {
            float4_t t = seg[mt][nt];
            if (started) {
                const float4_t o = tl[wave][mt * NT + nt][lane];
#pragma unroll
                for (int e = 0; e < 4; e++) t[e] = o[e] + seg[mt][nt][e];
            }
#pragma unroll
            for (int e = 0; e < 4; e++)
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(t[e]), ro,
                                                      vo + (((mt0 + mt) * 16 + e) * N + tile * 16) * 4, 0, 0);
        }
    }
}

// k_gemm_tm_sum: k_gemm_tm over every plane of its pairs and rows in one
// workgroup, unit by unit in K order. Each plane is finished as k_gemm_tm
// finishes it (the same segments and folds), and the finished planes are
// added in plane order into the one plane it writes: the sum every consumer
// forms from the P planes (in order from plane 0; those that pad with zero
// loads pad this sum the same way when P < 16), so the bits are the same,
// and the P-plane write and read are spared. For rows enough to fill the
// GPU without the K split (gemm_planes).
template <bool F32S>
__global__ __launch_bounds__(64 * TM_WAVES) void k_gemm_tm_sum(const uint8_t* __restrict__ Wr,
                                                              const uint4* __restrict__ Xp, int xp_mtiles,
                                                              float* __restrict__ out, int KU, int M, int N, int Nt,
                                                              int P, int Gm) {
    constexpr int NT = 2, R = TM_R, PW = R - 1, MTL = TM_MT, MTW = MTL * TM_PAIRS / TM_WAVES;
    static_assert(MTW * TM_WAVES == MTL * TM_PAIRS, "waves cover pairs x m-tiles");
    __shared__ u32x4 xs[2][MTL * 4][64];   // two units: block (m-tile, q = 2h + hl) of 1 KiB
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int npairs = Nt / NT;
    // Each pair group goes to one XCD, which runs its row blocks back to back
    // (the mapping of k_gemm_tm with one plane).
    const int nrb = (M + 16 * MTL - 1) / (16 * MTL), npg = (npairs + TM_PAIRS - 1) / TM_PAIRS;
    const int kx = blockIdx.x / 8;
    const int gx = (kx / nrb) * 8 + blockIdx.x % 8, gy = kx % nrb;
    if (gx >= npg) return;   // the grid is rounded up to whole XCD rounds
    const int pb = gx;
    const int pair = pb * TM_PAIRS + wave % TM_PAIRS, mw = (wave / TM_PAIRS) * MTW;   // m-tiles mw .. mw+MTW-1
    const bool has = pair < npairs;
    const int ua = 0, len = KU;   // every unit, planes in order
    const int mt0 = gy * MTL;
    const int G2 = 2 * KU;
    const auto rw = __builtin_amdgcn_make_buffer_rsrc((void*)Wr, 0, 0x7fffffff, 0x00020000);
    // activation m-tiles past the operand's allocation read zero
    const uint32_t xbytes = (uint32_t)min((unsigned long long)xp_mtiles * G2 * 2048ull, 0xffffffffull);
    const auto rx = __builtin_amdgcn_make_buffer_rsrc((void*)Xp, 0, xbytes, 0x00020000);
    const auto ro = __builtin_amdgcn_make_buffer_rsrc((void*)out, 0, M * N * 4, 0x00020000);
    const int vw = lane * 16, vs = NT * 1024 + (lane & 15) * NT * 4;
    const int vo = (4 * (lane >> 4) * N + (lane & 15)) * 4;
    const int pr0 = has ? pair : 0;
    // the load cursor (units are loaded in increasing order, PW ahead of
    // compute): the plane holding the next unit to load and its first record
    int lp = 0, lend = lx_plane_start(1, KU, P), lbase = 0, lrec = pr0 * lend * LX_REC;
    // the compute cursor: the plane being summed, its end and cut points
    int cp = 0, cbase = 0, cend = lend;
    uint32_t cuts = has ? lx_cuts(pair, npairs, Gm, cend) : 0u;

    // this wave's share of a unit's activations: blocks BPW*wave .. +BPW-1
    constexpr int BPW = MTL * 4 / TM_WAVES;
    static_assert(BPW * TM_WAVES == MTL * 4, "activation blocks split evenly over the waves");
    u32x4 st[BPW];
    auto load_x = [&](int u) {
        const int Uk = ua + (u < len ? u : len - 1);
#pragma unroll
        for (int k = 0; k < BPW; k++) {
            const int b = BPW * wave + k, mt = b >> 2, q = b & 3;
            const int src = ((mt0 + mt) * G2 + 2 * Uk + (q >> 1)) * 2 + (q & 1);
            st[k] = __builtin_amdgcn_raw_buffer_load_b128(rx, vw, src * 1024, 0);
        }
    };
    auto store_x = [&](int buf) {
#pragma unroll
        for (int k = 0; k < BPW; k++) xs[buf][BPW * wave + k][lane] = st[k];
    };
    u32x4 w[R][NT];
    uint32_t sc[R][NT];
    auto load_w = [&](int u, u32x4 (&wv)[NT], uint32_t (&sv)[NT]) {
        u = u < len ? u : len - 1;
        while (u >= lend) {   // the next plane: records [plane][pair][unit]
            lp++;
            lbase = lend;
            lend = lx_plane_start(lp + 1, KU, P);
            lrec = (lbase * npairs + pr0 * (lend - lbase)) * LX_REC;
        }
        const int off = lrec + (u - lbase) * LX_REC;
        wv[0] = __builtin_amdgcn_raw_buffer_load_b128(rw, vw, off, 2);
        wv[1] = __builtin_amdgcn_raw_buffer_load_b128(rw, vw, off + 1024, 2);
        const auto s2 = __builtin_amdgcn_raw_buffer_load_b64(rw, vs, off, 0);
        sv[0] = s2[0];
        sv[1] = s2[1];
    };
    float4_t seg[MTW][NT], tot[MTW][NT], sum[MTW][NT];
#pragma unroll
    for (int mt = 0; mt < MTW; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) seg[mt][nt] = tot[mt][nt] = sum[mt][nt] = float4_t{0.f, 0.f, 0.f, 0.f};
    bool started = false;   // tot holds the first segment(s)

    load_x(0);
#pragma unroll
    for (int i = 0; i < PW; i++) load_w(i, w[i], sc[i]);
    store_x(0);
    load_x(1);
    __syncthreads();

    auto unit = [&](int u, const u32x4 (&wc)[NT], const uint32_t (&sv)[NT]) {
        const int buf = u & 1;
        // the unit k_gemm_lx begins a new partial sum at: fold the running one
        if ((cuts >> (u - cbase)) & 1u) {
#pragma unroll
            for (int mt = 0; mt < MTW; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++) {
                    if (started)
#pragma unroll
                        for (int e = 0; e < 4; e++) tot[mt][nt][e] = tot[mt][nt][e] + seg[mt][nt][e];
                    else
                        tot[mt][nt] = seg[mt][nt];
                    seg[mt][nt] = float4_t{0.f, 0.f, 0.f, 0.f};
                }
            started = true;
        }
        half8_t b[2][NT], bl[2][NT];   // bl: the lo half's fragment, 2^-11 b
        float scale[2][NT];
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                b[h][nt] = h ? dequant8_biased(wc[nt][2], wc[nt][3]) : dequant8_biased(wc[nt][0], wc[nt][1]);
                bl[h][nt] = lo_weight8(b[h][nt]);
                scale[h][nt] = rec_scale<F32S>(sv[nt], h);
            }
        // per half-group, every m-tile's MFMA pair first and the scale FMAs
        // after them, so no FMA waits on the MFMA issued just before it; each
        // output's operations and their order are those of k_gemm_lx
#pragma unroll
        for (int h = 0; h < 2; h++) {
            u32x4 xv[MTW][2];
#pragma unroll
            for (int mt = 0; mt < MTW; mt++)
#pragma unroll
                for (int q = 0; q < 2; q++) xv[mt][q] = xs[buf][(mw + mt) * 4 + 2 * h + q][lane];
            float4_t pp[MTW][NT];
#pragma unroll
            for (int mt = 0; mt < MTW; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
                    pp[mt][nt] = mfma16x16x32(__builtin_bit_cast(half8_t, xv[mt][0]), b[h][nt], float4_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int mt = 0; mt < MTW; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
                    pp[mt][nt] = mfma16x16x32(__builtin_bit_cast(half8_t, xv[mt][1]), bl[h][nt], pp[mt][nt]);
#pragma unroll
            for (int mt = 0; mt < MTW; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
#pragma unroll
                    for (int e = 0; e < 4; e++) seg[mt][nt][e] = __builtin_fmaf(scale[h][nt], pp[mt][nt][e], seg[mt][nt][e]);
        }
        if (u + 1 == cend) {   // the plane's value (its last segment folded in) joins the sum
#pragma unroll
            for (int mt = 0; mt < MTW; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++) {
                    float4_t v = seg[mt][nt];
                    if (started)
#pragma unroll
                        for (int e = 0; e < 4; e++) v[e] = tot[mt][nt][e] + seg[mt][nt][e];
                    if (cp == 0)
                        sum[mt][nt] = v;
                    else
#pragma unroll
                        for (int e = 0; e < 4; e++) sum[mt][nt][e] = sum[mt][nt][e] + v[e];
                    seg[mt][nt] = float4_t{0.f, 0.f, 0.f, 0.f};
                }
            started = false;
            if (cp + 1 < P) {
                cp++;
                cbase = cend;
                cend = lx_plane_start(cp + 1, KU, P);
                cuts = has ? lx_cuts(pair, npairs, Gm, cend - cbase) : 0u;
            }
        }
    };
    int u = 0;
    for (; u + R <= len; u += R) {
#pragma unroll
        for (int I = 0; I < R; I++) {
            load_w(u + I + PW, w[(I + PW) % R], sc[(I + PW) % R]);
            unit(u + I, w[I], sc[I]);
            // the next unit's activations go in the other buffer: every wave
            // finished reading it (one unit ago) before the last barrier
            store_x((I + 1) & 1);
            load_x(u + I + 2);
            __syncthreads();
        }
    }
    // at most PW units remain, their records in ring slots 0 .. PW-1
#pragma unroll
    for (int I = 0; I < PW; I++) {
        if (u + I < len) {
            unit(u + I, w[I], sc[I]);
            store_x((I + 1) & 1);
            load_x(u + I + 2);
            __syncthreads();
        }
    }
    if (!has) return;
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        const int tile = pair * NT + nt;
        if (tile * 16 >= N) continue;
        if (tile * 16 + 16 > N && tile * 16 + (lane & 15) >= N) continue;
#pragma unroll
        for (int mt = 0; mt < MTW; mt++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(sum[mt][nt][e]), ro,
                                                      vo + (((mt0 + mw + mt) * 16 + e) * N + tile * 16) * 4, 0, 0);
    }
}

// The planes launch_gemm writes for w at M rows: w.P, or one when the many
// rows give every CU two workgroups or more without the K split
// (k_gemm_tm_sum, 2 <= P < 16).
int gemm_planes(const QTensor& w, int M, int ncu) {
    if (M <= 32 || w.P < 2 || w.P >= 16) return w.P;
    const long long work = (long long)((w.Nt / 2 + TM_PAIRS - 1) / TM_PAIRS) * ((M + 16 * TM_MT - 1) / (16 * TM_MT));
    return work >= 2LL * ncu ? 1 : w.P;
}

template <bool F32S>
static void launch_gemm_fmt(hipStream_t st, const QTensor& w, const uint4* Xp, int xp_mtiles, float* out, int M,
                            int ncu) {
    if (M <= 16) launch_lx<1, F32S>(st, w, Xp, out, M, ncu);
    else if (M <= 32) launch_lx<2, F32S>(st, w, Xp, out, M, ncu);
    else {
        // the same planes and cut points as k_gemm_lx (lx_groups)
        const int Gm = lx_groups(w, ncu) / w.P;
        const int npairs = w.Nt / 2;
        const bool sum = gemm_planes(w, M, ncu) == 1;
        const int nrb = (M + 16 * TM_MT - 1) / (16 * TM_MT);
        // Twelve pairs a workgroup where that takes fewer rounds of
        // workgroups over the CUs, counting a round of the twelve-wave kernel
        // as 1.5 of the eight-wave one's (measured at 128 rows: 39 against
        // 25 us a round at gate|up, 36 against 25 at down): at 128 rows
        // gate|up runs 3 rounds instead of 5 and down 2 instead of 3.
        const int units12 = w.P * ((npairs + TM12_WAVES - 1) / TM12_WAVES);
        const long long r8 = ((long long)w.P * ((npairs + TM_PAIRS - 1) / TM_PAIRS) * nrb + ncu - 1) / ncu;
        const long long r12 = ((long long)units12 * nrb + ncu - 1) / ncu;
        if (!sum && 3 * r12 <= 2 * r8) {
            dim3 grid(8 * ((units12 + 7) / 8) * nrb);
            hipLaunchKernelGGL(k_gemm_tm12<F32S>, grid, dim3(64 * TM12_WAVES), 0, st, (const uint8_t*)w.codes, Xp,
                               xp_mtiles, out, w.KU, M, w.N, w.Nt, w.P, Gm);
            CHECK_LAUNCH();
            return;
        }
        const int units = (sum ? 1 : w.P) * ((npairs + TM_PAIRS - 1) / TM_PAIRS);
        dim3 grid(8 * ((units + 7) / 8) * nrb);
        if (sum)
            hipLaunchKernelGGL(k_gemm_tm_sum<F32S>, grid, dim3(64 * TM_WAVES), 0, st, (const uint8_t*)w.codes, Xp,
                               xp_mtiles, out, w.KU, M, w.N, w.Nt, w.P, Gm);
        else
            hipLaunchKernelGGL(k_gemm_tm<F32S>, grid, dim3(64 * TM_WAVES), 0, st, (const uint8_t*)w.codes, Xp,
                               xp_mtiles, out, w.KU, M, w.N, w.Nt, w.P, Gm);
    }
    CHECK_LAUNCH();
}

void launch_gemm(hipStream_t st, const QTensor& w, const uint4* Xp, int xp_mtiles, float* out, int M, int ncu) {
    if (w.f32s) launch_gemm_fmt<true>(st, w, Xp, xp_mtiles, out, M, ncu);
    else launch_gemm_fmt<false>(st, w, Xp, xp_mtiles, out, M, ncu);
}

// =========================================================== operand prep ===
// Writes 8 consecutive values of row m (columns 8c .. 8c+7) as the f16 hi/lo
// operand fragments of the GEMM (layout above; lo scaled by 2^11).
__device__ static inline void write_hilo(uint4* Xp, int m, int c, int KU, const float* v) {
    const int g = c >> 2, kb = c & 3;
    const int mt = m >> 4, lane = (m & 15) + 16 * kb;
    half8_t hi, lo;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        _Float16 a, b;
        split_hilo_x(v[j], a, b);
        hi[j] = a;
        lo[j] = b;
    }
    const size_t at = (((size_t)mt * 2 * KU + g) * 2) * 64 + lane;
    Xp[at] = __builtin_bit_cast(uint4, hi);
    Xp[at + 64] = __builtin_bit_cast(uint4, lo);
}

__global__ void k_prep_rows(const float* __restrict__ x, int ldx, int M, int Mpad, int K, int KU,
                            uint4* __restrict__ Xp) {
    const int per = 8 * KU;
    const int total = Mpad * per;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
        const int m = i / per, c = i % per;
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int k = 8 * c + j;
            v[j] = (m < M && k < K) ? x[(size_t)m * ldx + k] : 0.0f;
        }
        write_hilo(Xp, m, c, KU, v);
    }
}

void launch_prep_rows(hipStream_t st, const float* x, int ldx, int M, int Mpad, int K, int KU,
                      uint4* Xp) {
    const int total = Mpad * 8 * KU;
    hipLaunchKernelGGL(k_prep_rows, dim3((total + 255) / 256), dim3(256), 0, st, x, ldx, M, Mpad, K, KU, Xp);
    CHECK_LAUNCH();
}

// ========================================================= finish kernels ===
// Residual step and rmsnorm, one workgroup of 1024 threads per row, the row
// held in registers (4 columns a thread per pass, H <= 8192):
//   x = x + the projection's K planes added in order (add_inplace,
//   web/model/kernels.js:1334-1346), optionally round_f16 (:1356-1383, the
//   per-block residual round, model.js:619-624), written back;
//   then, with w: rmsnorm (:930-976), y = x * (1/sqrt(ss/H + eps)) * w, as the
//   next matmul's f16 hi/lo operand Xp (or as rows y). ss is summed per wave
//   (butterfly) and then over the waves in order.
// part == nullptr: the x rows as they are, gathered through `rows` (the entry
// rows, the head's sampled rows). Rows M .. Mpad-1 get zero operand rows.
constexpr int RN_THREADS = 1024, RN_PASSES = 2, RN_SPLITS = 16;
__global__ __launch_bounds__(RN_THREADS) void k_resid_norm(float* __restrict__ x, const int32_t* __restrict__ rows,
                                                           const float* __restrict__ part, int splits, int M, int H,
                                                           int round, const float* __restrict__ w, float eps, int KU,
                                                           uint4* __restrict__ Xp, float* __restrict__ y) {
    __shared__ float red[RN_THREADS / 64];
    __shared__ float scale_s;
    const int m = blockIdx.x, t = threadIdx.x, lane = t & 63;
    const int n4 = H >> 2;
    if (m >= M) {
        const float z[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        for (int c8 = t; c8 < 8 * KU; c8 += RN_THREADS) write_hilo(Xp, m, c8, KU, z);
        return;
    }
    const size_t xoff = (size_t)(rows ? rows[m] : m) * H;
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 v[RN_PASSES], wv[RN_PASSES];
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < RN_PASSES; k++) {
        const int c4 = t + k * RN_THREADS;
        v[k] = wv[k] = zero;
        if (c4 >= n4) continue;
        if (w) wv[k] = *(const float4*)(w + 4 * c4);   // in flight with the row's loads
        float4 xv = *(const float4*)(x + xoff + 4 * c4);
        if (part) {
            // every plane's load in flight at once, through a resource sized
            // to the planes: a load past the last one reads zero (no branch),
            // and adding +0 leaves the in-order sum as it is
            const auto rp = __builtin_amdgcn_make_buffer_rsrc((void*)part, 0, splits * M * H * 4, 0x00020000);
            float4 pv[RN_SPLITS];
#pragma unroll
            for (int s = 0; s < RN_SPLITS; s++) {
                const u32x4 q = __builtin_amdgcn_raw_buffer_load_b128(rp, (m * H + 4 * c4) * 4, s * M * H * 4, 0);
                pv[s] = make_float4(__uint_as_float(q[0]), __uint_as_float(q[1]), __uint_as_float(q[2]),
                                    __uint_as_float(q[3]));
            }
            float4 p = pv[0];
#pragma unroll
            for (int s = 1; s < RN_SPLITS; s++)
                p = make_float4(p.x + pv[s].x, p.y + pv[s].y, p.z + pv[s].z, p.w + pv[s].w);
            for (int s = RN_SPLITS; s < splits; s++) {
                const float4 q = *(const float4*)(part + ((size_t)s * M + m) * H + 4 * c4);
                p = make_float4(p.x + q.x, p.y + q.y, p.z + q.z, p.w + q.w);
            }
            xv = make_float4(xv.x + p.x, xv.y + p.y, xv.z + p.z, xv.w + p.w);
            if (round)
                xv = make_float4(round_f16_value(xv.x), round_f16_value(xv.y), round_f16_value(xv.z),
                                 round_f16_value(xv.w));
            *(float4*)(x + xoff + 4 * c4) = xv;
        }
        v[k] = xv;
        ss = ss + xv.x * xv.x;
        ss = ss + xv.y * xv.y;
        ss = ss + xv.z * xv.z;
        ss = ss + xv.w * xv.w;
    }
    if (!w) return;   // the residual step alone (the pass's last block)
    ss = wave_sum(ss);
    if (lane == 0) red[t >> 6] = ss;
    __syncthreads();
    if (t == 0) {
        float tot = 0.0f;
        for (int i = 0; i < RN_THREADS / 64; i++) tot = tot + red[i];
        scale_s = 1.0f / sqrtf(tot / (float)H + eps);
    }
    __syncthreads();
    const float scale = scale_s;
#pragma unroll
    for (int k = 0; k < RN_PASSES; k++) {
        const int c4 = t + k * RN_THREADS;
        float o[4] = {0.f, 0.f, 0.f, 0.f};
        if (c4 < n4) {
            o[0] = v[k].x * scale * wv[k].x;
            o[1] = v[k].y * scale * wv[k].y;
            o[2] = v[k].z * scale * wv[k].z;
            o[3] = v[k].w * scale * wv[k].w;
            if (y) *(float4*)(y + (size_t)m * H + 4 * c4) = make_float4(o[0], o[1], o[2], o[3]);
        }
        if (Xp) {
            // lanes (2i, 2i+1) hold the two halves of one 8-column operand chunk
            float e[8];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                e[q] = o[q];
                e[4 + q] = __shfl_xor(o[q], 1);
            }
            if (c4 < n4 && (c4 & 1) == 0) write_hilo(Xp, m, c4 >> 1, KU, e);
        }
    }
    if (Xp) {
        // operand columns past H (K padded to whole 64-column units)
        const float z[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        for (int c8 = (H >> 3) + t; c8 < 8 * KU; c8 += RN_THREADS) write_hilo(Xp, m, c8, KU, z);
    }
}

void launch_resid_norm(hipStream_t st, float* x, const int32_t* rows, const float* part, int splits, int M, int Mpad,
                       int H, int round, const float* w, float eps, int KU, uint4* Xp, float* y) {
    hipLaunchKernelGGL(k_resid_norm, dim3(Xp ? Mpad : M), dim3(RN_THREADS), 0, st, x, rows, part, splits, M, H, round,
                       w, eps, KU, Xp, y);
    CHECK_LAUNCH();
}

// rmsnorm (web/model/kernels.js:930-976) is y = x * f * w with the row factor
// f = 1/sqrt(ss/H + eps); the matmul that follows is linear in its operand,
// so (x*f*w) . W^T = f * ((x*w) . W^T). The residual kernel below writes the
// operand x*w and the row's partial sums of squares; the matmul's consumer
// multiplies the summed planes by f (row_scale). This takes the row-wide
// reduction off the path between the residual step and the matmul, so the
// residual step spreads over (slice, row) workgroups instead of one per row.
// In two parts, so a caller can issue the loads beside its own:
// row_scale_load puts all RW_SMAX loads of row m in flight at once (the
// resource's base is the array's, uniform for any m; the slots past the nsl
// partials read as zero), row_scale_of adds them in order.
struct RowSS {
    float q[RW_SMAX];
};
__device__ static inline RowSS row_scale_load(const RowScale& rs, int m) {
    RowSS r;
    if (!rs.ssp) return r;
    const auto rq = __builtin_amdgcn_make_buffer_rsrc((void*)rs.ssp, 0, 0x7fffffff, 0x00020000);
#pragma unroll
    for (int s = 0; s < RW_SMAX; s++) {
        const float v = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rq, (m * RW_SMAX + s) * 4, 0, 0));
        r.q[s] = s < rs.nsl ? v : 0.0f;
    }
    return r;
}
__device__ static inline float row_scale_of(const RowScale& rs, const RowSS& r) {
    if (!rs.ssp) return 1.0f;
    float tot = 0.0f;
#pragma unroll
    for (int s = 0; s < RW_SMAX; s++) tot = tot + r.q[s];
    return 1.0f / sqrtf(tot / (float)rs.H + rs.eps);
}
__device__ static inline float row_scale(const RowScale& rs, int m) { return row_scale_of(rs, row_scale_load(rs, m)); }

// Residual step (add_inplace, web/model/kernels.js:1334-1346: x plus the
// projection's planes added in order; optional round_f16, :1356-1383, the
// per-block round of model.js:619-624), then, with w, the next matmul's
// operand x*w as f16 hi/lo and this slice's sum of squares of x (each
// thread's 4 values in order, a wave butterfly, the two waves in order) at
// ssp[m*RW_SMAX + slice]. Workgroup (slice, row): 128 threads, a float4 of
// the row each. part == nullptr: x as it is. Rows M .. Mpad-1 get zero
// operand rows. H % 64 == 0, so the operand has no padding columns. SP plane
// loads are issued at once (4 when the projection has at most 4 planes, so
// no load goes out past them; 16 otherwise), the rest in a loop.
template <int SP>
__global__ __launch_bounds__(RW_THREADS) void k_resid_w(const float* x, float* xo, const float* __restrict__ part,
                                                      int splits, int M, int H, int round,
                                                      const float* __restrict__ w, int KU, uint4* __restrict__ Xp,
                                                      float* __restrict__ ssp) {
    __shared__ float red[RW_THREADS / 64];
    const int m = blockIdx.y, sl = blockIdx.x, t = threadIdx.x, lane = t & 63;
    const int n4 = H >> 2, c4 = sl * RW_THREADS + t;
    const bool live = c4 < n4;
    if (m >= M) {
        if (Xp && live && (c4 & 1) == 0) {
            const float z[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            write_hilo(Xp, m, c4 >> 1, KU, z);
        }
        return;
    }
    const size_t xoff = (size_t)m * H + 4 * (size_t)c4;
    float4 xv = make_float4(0.f, 0.f, 0.f, 0.f), wv = xv;
    if (live) {
        if (w) wv = *(const float4*)(w + 4 * c4);
        xv = *(const float4*)(x + xoff);
        if (part) {
            // every plane's load in flight at once, through a resource sized
            // to the planes: a load past the last one reads zero (no branch),
            // and adding +0 leaves the in-order sum as it is
            const auto rp = __builtin_amdgcn_make_buffer_rsrc((void*)part, 0, splits * M * H * 4, 0x00020000);
            float4 pv[SP];
#pragma unroll
            for (int s = 0; s < SP; s++) {
                const u32x4 q = __builtin_amdgcn_raw_buffer_load_b128(rp, (int)xoff * 4, s * M * H * 4, 0);
                pv[s] = make_float4(__uint_as_float(q[0]), __uint_as_float(q[1]), __uint_as_float(q[2]),
                                    __uint_as_float(q[3]));
            }
            float4 pp = pv[0];
#pragma unroll
            for (int s = 1; s < SP; s++)
                pp = make_float4(pp.x + pv[s].x, pp.y + pv[s].y, pp.z + pv[s].z, pp.w + pv[s].w);
            for (int s = SP; s < splits; s++) {
                const float4 q = *(const float4*)(part + (size_t)s * M * H + xoff);
                pp = make_float4(pp.x + q.x, pp.y + q.y, pp.z + q.z, pp.w + q.w);
            }
            xv = make_float4(xv.x + pp.x, xv.y + pp.y, xv.z + pp.z, xv.w + pp.w);
            if (round)
                xv = make_float4(round_f16_value(xv.x), round_f16_value(xv.y), round_f16_value(xv.z),
                                 round_f16_value(xv.w));
            *(float4*)(xo + xoff) = xv;
        }
    }
    if (!w) return;   // the residual step alone (the pass's last block)
    float ss = 0.0f;
    ss = ss + xv.x * xv.x;
    ss = ss + xv.y * xv.y;
    ss = ss + xv.z * xv.z;
    ss = ss + xv.w * xv.w;
    ss = wave_sum(ss);
    if (lane == 0) red[t >> 6] = ss;
    // lanes (2i, 2i+1) hold the two halves of one 8-column operand chunk
    float o[4] = {xv.x * wv.x, xv.y * wv.y, xv.z * wv.z, xv.w * wv.w};
    float e[8];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        e[q] = o[q];
        e[4 + q] = __shfl_xor(o[q], 1);
    }
    if (live && (c4 & 1) == 0) write_hilo(Xp, m, c4 >> 1, KU, e);
    __syncthreads();
    if (t == 0) {
        float tot = 0.0f;
        for (int i = 0; i < RW_THREADS / 64; i++) tot = tot + red[i];
        ssp[(size_t)m * RW_SMAX + sl] = tot;
    }
}

void launch_resid_w(hipStream_t st, const float* x, float* xo, const float* part, int splits, int M, int Mpad, int H,
                    int round, const float* w, int KU, uint4* Xp, float* ssp) {
    const int nsl = (H / 4 + RW_THREADS - 1) / RW_THREADS;
    const dim3 grid(nsl, w ? Mpad : M);
    if (splits <= 4)
        hipLaunchKernelGGL(k_resid_w<4>, grid, dim3(RW_THREADS), 0, st, x, xo, part, splits, M, H, round, w, KU, Xp,
                           ssp);
    else
        hipLaunchKernelGGL(k_resid_w<RN_SPLITS>, grid, dim3(RW_THREADS), 0, st, x, xo, part, splits, M, H, round, w,
                           KU, Xp, ssp);
    CHECK_LAUNCH();
}

// The residual step of k_resid_w on N columns of row m from column k0 (N and
// k0 multiples of 4): x plus the planes in order, rounded on demand. Its
// kernels pad the plane sum with +0 to 4 or 16 planes, which turns a sum of
// -0 into +0: so does this one.
template <int N>
__device__ static inline void resid_row(const LxPro& p, int M, int H, int m, int k0, float (&x)[N]) {
    const auto rp = __builtin_amdgcn_make_buffer_rsrc((void*)p.part, 0, p.splits * M * H * 4, 0x00020000);
    const int at = (m * H + k0) * 4, plane = M * H * 4;
    float s[N];
#pragma unroll
    for (int e = 0; e < N; e += 4) {
        const float4 v = *(const float4*)(p.x + (size_t)m * H + k0 + e);
        x[e] = v.x; x[e + 1] = v.y; x[e + 2] = v.z; x[e + 3] = v.w;
        s[e] = s[e + 1] = s[e + 2] = s[e + 3] = 0.0f;
    }
    for (int q = 0; q < p.splits; q += 4) {   // four planes' loads in flight; past the last one a load reads +0
        u32x4 v[4][N / 4];
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int e = 0; e < N / 4; e++) v[i][e] = __builtin_amdgcn_raw_buffer_load_b128(rp, at + 16 * e, (q + i) * plane, 0);
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int e = 0; e < N; e++) {
                const float f = __uint_as_float(v[i][e / 4][e % 4]);
                s[e] = q + i == 0 ? f : s[e] + f;
            }
    }
#pragma unroll
    for (int e = 0; e < N; e++) {
        if (p.splits > 4 && p.splits < 16) s[e] = s[e] + 0.0f;
        x[e] = x[e] + s[e];
        if (p.round) x[e] = round_f16_value(x[e]);
    }
}

// The rest of k_resid_w for four (slice, row) pairs: the new rows to xo and
// the slices' sums of squares. 128 threads a pair; red: 2 floats a pair.
__device__ static void resid_slices(const LxPro& p, int M, int H, float* red) {
    const int t = threadIdx.x % RW_THREADS, g = threadIdx.x / RW_THREADS, lane = t & 63;
    const int nsl = (H / 4 + RW_THREADS - 1) / RW_THREADS;
    const int i = (blockIdx.x - p.G) * 4 + g, m = i / nsl, sl = i % nsl;
    const int c4 = sl * RW_THREADS + t;
    const bool live = m < M && c4 < H / 4;
    float x[4] = {0.f, 0.f, 0.f, 0.f};
    if (live) {
        resid_row<4>(p, M, H, m, 4 * c4, x);
        *(float4*)(p.xo + (size_t)m * H + 4 * c4) = make_float4(x[0], x[1], x[2], x[3]);
    }
    float ss = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; e++) ss = ss + x[e] * x[e];
    ss = wave_sum(ss);
    if (lane == 0) red[2 * g + (t >> 6)] = ss;
    __syncthreads();
    if (t == 0 && m < M) p.ssp[(size_t)m * RW_SMAX + sl] = (0.0f + red[2 * g]) + red[2 * g + 1];
}

// k_fin_swiglu's 8 columns of row m from column k0, with the row factor f.
__device__ static inline void swiglu8(const LxPro& p, int M, int m, int k0, float f, float (&v)[8]) {
    const size_t N2 = 2 * (size_t)p.F, plane = (size_t)M * N2;
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = 0.0f;
    if (k0 >= p.F) return;   // F is a multiple of 32: 8 columns are in or out together
    float g[8], u[8];
    const auto rp = __builtin_amdgcn_make_buffer_rsrc((void*)p.part, 0, (uint32_t)(p.splits * plane * 4), 0x00020000);
    const int at = (int)(((size_t)m * N2 + k0) * 4);
    for (int q = 0; q < p.splits; q += 4) {
        u32x4 x[4][4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int so = (int)((q + i) * plane * 4);
            x[i][0] = __builtin_amdgcn_raw_buffer_load_b128(rp, at, so, 0);
            x[i][1] = __builtin_amdgcn_raw_buffer_load_b128(rp, at + 16, so, 0);
            x[i][2] = __builtin_amdgcn_raw_buffer_load_b128(rp, at + 4 * p.F, so, 0);
            x[i][3] = __builtin_amdgcn_raw_buffer_load_b128(rp, at + 4 * p.F + 16, so, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (q + i < p.splits)
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float a = __uint_as_float(x[i][e >> 2][e & 3]), b = __uint_as_float(x[i][2 + (e >> 2)][e & 3]);
                    g[e] = q + i == 0 ? a : g[e] + a;
                    u[e] = q + i == 0 ? b : u[e] + b;
                }
    }
#pragma unroll
    for (int e = 0; e < 8; e++) {
        g[e] = g[e] * f;
        u[e] = u[e] * f;
        const float sc = 1.0f / (1.0f + expf(-g[e]));
        v[e] = g[e] * sc * u[e];
    }
}

// Whether w's matmul at M rows forms its operand itself: yes while what each
// workgroup then reads, its columns of `values` f32 planes of M rows, is at
// most this. Reading it is the cost: a launch saved is about 3 us, and a
// workgroup's share comes in at about 100 KB/us once the launch's others (one
// a CU at most) read theirs from the L2s too. Passes measured with the line swept from 0 to 4 MB,
// none fused against the best line against every one fused, us:
//   hidden 576,  8 blocks:  1 row 384/313/313, 4: 388/325/326, 16: 414/375/375
//   hidden 4096, 4 blocks:  1 row 368/334/334, 4: 384/364/365, 8: 401/395/401,
//                           12: 417/415/436, 16: 433/433/469
//   hidden 5120, 3 blocks:  1 row 348/319/319, 4: 360/348/349, 8: 379/375/381,
//                           12: 395/395/417, 16: 411/411/449
// The best line is 256 KB in every one of them, to within their noise of
// 0.3%; at 384 KB and past it the passes of 8 to 16 rows lose.
constexpr size_t LX_PRO_BYTES = 256 << 10;
bool gemm_fuses(const QTensor& w, int M, int values) {
    const int len = (w.KU + w.P - 1) / w.P;
    return M <= GEMM_FUSE_ROWS && (size_t)M * values * len * 256 <= LX_PRO_BYTES;
}

void launch_gemm_resid(hipStream_t st, const QTensor& w, const float* x, float* xo, const float* part, int splits,
                       int round, const float* norm, float* ssp, float* out, int M, int ncu) {
    LxPro p;
    p.part = part;
    p.splits = splits;
    p.x = x;
    p.xo = xo;
    p.w = norm;
    p.round = round;
    p.ssp = ssp;
    if (w.f32s) launch_lx<1, true, LX_PRO_RESID>(st, w, nullptr, out, M, ncu, p);
    else launch_lx<1, false, LX_PRO_RESID>(st, w, nullptr, out, M, ncu, p);
    CHECK_LAUNCH();
}

void launch_gemm_swiglu(hipStream_t st, const QTensor& w, const float* part, int splits, int F, const RowScale& rs,
                        float* out, int M, int ncu) {
    LxPro p;
    p.part = part;
    p.splits = splits;
    p.rs = rs;
    p.F = F;
    if (w.f32s) launch_lx<1, true, LX_PRO_SWIGLU>(st, w, nullptr, out, M, ncu, p);
    else launch_lx<1, false, LX_PRO_SWIGLU>(st, w, nullptr, out, M, ncu, p);
    CHECK_LAUNCH();
}

// SwiGLU (web/model/kernels.js:1513-1529 silu_mul): act = g * (1/(1+exp(-g)))
// * up over the fused gate|up projection, straight into the down operand.
// SP > 0: at most SP planes, every plane's loads issued at once (through a
// resource sized to the planes, so those past the last read zero and are not
// added), before the row factor's; SP = 0: any plane count, in a loop.
template <int SP>
__global__ __launch_bounds__(256) void k_fin_swiglu(const float* __restrict__ part, int splits, int M, int Mpad,
                                                    int F, int KU, uint4* __restrict__ Xp, RowScale rs) {
    // one thread per (row, 8 columns); the planes are added in order
    const int per = 8 * KU;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= Mpad * per) return;
    const int m = i / per, c = i % per, k0 = 8 * c;
    const size_t N2 = 2 * (size_t)F, plane = (size_t)M * N2;
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (m < M && k0 < F) {
        float g[8], u[8];
        const float* row = part + (size_t)m * N2 + k0;
        const bool fast = k0 + 8 <= F && (F & 3) == 0;
        u32x4 q[SP > 0 ? SP : 1][4];
        if constexpr (SP > 0) {
            // issued by every thread (no branch to join): a thread off the fast
            // path reads in-bounds or zero values it does not use
            const auto rp = __builtin_amdgcn_make_buffer_rsrc((void*)part, 0, (uint32_t)(splits * plane * 4),
                                                              0x00020000);
            const int at = (int)(((size_t)m * N2 + k0) * 4);
#pragma unroll
            for (int s = 0; s < SP; s++) {
                const int so = (int)(s * plane * 4);
                q[s][0] = __builtin_amdgcn_raw_buffer_load_b128(rp, at, so, 0);
                q[s][1] = __builtin_amdgcn_raw_buffer_load_b128(rp, at + 16, so, 0);
                q[s][2] = __builtin_amdgcn_raw_buffer_load_b128(rp, at + 4 * F, so, 0);
                q[s][3] = __builtin_amdgcn_raw_buffer_load_b128(rp, at + 4 * F + 16, so, 0);
            }
        }
        // the gate|up operand carried x*w: rmsnorm's row factor goes on below
        // (its loads issued here, after the planes')
        const RowSS rq = row_scale_load(rs, m);
        if (SP > 0 && fast) {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                g[j] = __uint_as_float(q[0][j >> 2][j & 3]);
                u[j] = __uint_as_float(q[0][2 + (j >> 2)][j & 3]);
            }
#pragma unroll
            for (int s = 1; s < SP; s++)
                if (s < splits)
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        g[j] = g[j] + __uint_as_float(q[s][j >> 2][j & 3]);
                        u[j] = u[j] + __uint_as_float(q[s][2 + (j >> 2)][j & 3]);
                    }
        } else if (fast) {
            auto ld8 = [&](const float* p, float* x) {
                const float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
                x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w; x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
            };
            ld8(row, g);
            ld8(row + F, u);
#pragma unroll 4
            for (int s = 1; s < splits; s++) {
                float gs[8], us[8];
                ld8(row + s * plane, gs);
                ld8(row + s * plane + F, us);
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    g[j] = g[j] + gs[j];
                    u[j] = u[j] + us[j];
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                g[j] = u[j] = 0.0f;
                if (k0 + j >= F) continue;
                g[j] = row[j];
                u[j] = row[F + j];
                for (int s = 1; s < splits; s++) {
                    g[j] = g[j] + row[s * plane + j];
                    u[j] = u[j] + row[s * plane + F + j];
                }
            }
        }
        const float f = row_scale_of(rs, rq);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            g[j] = g[j] * f;
            u[j] = u[j] * f;
        }
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float sc = 1.0f / (1.0f + expf(-g[j]));
            v[j] = k0 + j < F ? g[j] * sc * u[j] : 0.0f;
        }
    }
    write_hilo(Xp, m, c, KU, v);
}

void launch_fin_swiglu(hipStream_t st, const float* part, int splits, int M, int Mpad, int F, int KU,
                       uint4* Xp, const RowScale& rs) {
    const int total = Mpad * 8 * KU;
    const dim3 grid((total + 255) / 256);
    // the buffer resource's offsets are 32-bit
    const bool small = (size_t)splits * M * 2 * (size_t)F * 4 < (1ull << 31);
    if (small && splits <= 1)
        hipLaunchKernelGGL(k_fin_swiglu<1>, grid, dim3(256), 0, st, part, splits, M, Mpad, F, KU, Xp, rs);
    else if (small && splits <= 4)
        hipLaunchKernelGGL(k_fin_swiglu<4>, grid, dim3(256), 0, st, part, splits, M, Mpad, F, KU, Xp, rs);
    else
        hipLaunchKernelGGL(k_fin_swiglu<0>, grid, dim3(256), 0, st, part, splits, M, Mpad, F, KU, Xp, rs);
    CHECK_LAUNCH();
}

// ============================================================ KV geometry ===
// One (page, kv head) block of the pool, blk = 64*D + 64*ng*4 bytes:
//   K: codes [64 tokens][D] with column d at (D/4)*((d%32)/8) + 8*(d/32) + d%8,
//      so one lane's fragment bytes for every group are contiguous; then f32
//      scales [64 tokens][ng].
//   V: codes [4][D][16]: with v = vpos(s) = 16*((s%16)/4) + 4*(s/16) + s%4,
//      token s's code for channel d sits in 16-byte row (v/16, d) at byte
//      v%16, so a lane's P·V fragment (16 tokens of one channel) is one
//      contiguous 16-byte load, and one token's D codes lie in D*16 bytes
//      (a new token dirties 16 lines of 128 B at D = 128, not the 64 of a
//      [D][64] layout); then f32 scales [4][ng][16] at the same positions.
// Codes are stored biased (code ^ 0x80, i.e. code + 128) so the MFMA dequant
// puts them under an f16 exponent directly; they are the reference's store_kv
// codes bit for bit once converted back (k_kv_ref: cc_read_kv, cc_write_kv).
__host__ __device__ static inline int kpos(int d, int D) { return (D / 4) * ((d & 31) >> 3) + 8 * (d >> 5) + (d & 7); }
__host__ __device__ static inline int vpos(int s) { return 16 * ((s & 15) >> 2) + 4 * (s >> 4) + (s & 3); }
// byte of V code (channel d, token s) in its block, and float of V scale
// (group b, token s) after the codes
__host__ __device__ static inline int vcode_at(int d, int s, int D) {
    const int v = vpos(s);
    return ((v >> 4) * D + d) * 16 + (v & 15);
}
__host__ __device__ static inline int vscale_at(int b, int s, int ng) {
    const int v = vpos(s);
    return ((v >> 4) * ng + b) * 16 + (v & 15);
}

// store_kv (web/model/kernels.js:1024-1073) for a row's K and V, plus RoPE on
// its Q (kernels.js:1093-1129) into the attention operand, after the q|k|v
// splits are summed.
// Bit-exact with the reference given the same q|k|v row: RoPE a*cs - o*sn
// (no fused multiply-add: the build passes -ffp-contract=off), amax,
// scale = amax/127, inv = scale > 0 ? 1/scale : 0, rint, clamp ±127.
// Channel c of one head after split-half RoPE, given the (cos, sin) of c's
// pair at the row's position (tbl[(pos*(rot/2) + c mod rot/2)*2 + 0/1]);
// channels from rot on pass through.
__device__ static inline float rope_cs(const float* src, int c, int rot, float cs, float sn) {
    if (c >= rot) return src[c];
    const int half = rot >> 1;
    if (c < half) {
        const float a = src[c], o = src[c + half];
        return a * cs - o * sn;
    }
    const float a = src[c - half], o = src[c];
    return o * cs + a * sn;
}

// Spread over (row, head): one wave per head of a row, four heads per
// workgroup. The head's D values (K splits summed in order) sit in the wave's
// LDS slice; Q heads are RoPE'd into the attention operand, K heads RoPE'd and
// quantised into the pool, V heads quantised.
template <int D, int SU>
__global__ __launch_bounds__(256) void k_fin_qkv(const float* __restrict__ part, int splits, int M,
                                                  const int32_t* __restrict__ row_job,
                                                  const JobDev* __restrict__ jobs, int nH, int group, KVGeom g,
                                                  const float* __restrict__ tbl, int rot, uint8_t* __restrict__ kpool,
                                                  uint8_t* __restrict__ vpool,
                                                  const uint32_t* __restrict__ page_table, uint4* __restrict__ Qp,
                                                  RowScale rs, int do_q, int do_kv, QkExtras ex) {
    __shared__ float buf[4][D];
    __shared__ __attribute__((aligned(16))) float rq[4][D];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = blockIdx.y;
    const int nKV = g.nKV;
    const int nqkv = nH + 2 * nKV;
    const int nall = nqkv + (ex.gate ? nH : 0);   // a hybrid block's gate heads follow v
    const int hidx = blockIdx.x * 4 + wave;
    const bool live = hidx < nall;
    const int N = nall * D;
    // SU planes' loads in flight at once, first (4 when q|k|v has at most 4
    // planes, else 16), through a resource sized to the planes: past the last
    // one a load reads zero (no branch), and adding +0 leaves the in-order sum
    // as it is; planes past SU in a loop
    constexpr int DH = D / 64;
    float pv[DH][SU];
    if (live) {
        const auto rp = __builtin_amdgcn_make_buffer_rsrc((void*)part, 0, splits * M * N * 4, 0x00020000);
#pragma unroll
        for (int h = 0; h < DH; h++) {
            const int at = (m * N + hidx * D + 64 * h + lane) * 4;
#pragma unroll
            for (int s = 0; s < SU; s++)
                pv[h][s] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rp, at, s * M * N * 4, 0));
        }
    }
    // the row's job and its page, and rmsnorm's row factor (the q|k|v operand
    // carried x*w), looked up while the planes load
    const JobDev jb = jobs[row_job[m]];
    const int i = m - jb.row0;
    const int pos = jb.past + i;
    const uint32_t page = page_table[(size_t)jb.slot * g.max_pages + pos / g.page];
    const float f = row_scale(rs, m);
    // RoPE's (cos, sin) for this lane's channels 64h + lane at pos, loaded
    // here so they are in flight beside the planes
    float cs[DH], sn[DH];
    {
        const int half = rot >> 1;
#pragma unroll
        for (int h = 0; h < DH; h++) {
            const int c = 64 * h + lane;
            cs[h] = 1.0f;
            sn[h] = 0.0f;
            if (c < rot) {
                const float2 t2 = *(const float2*)(tbl + ((size_t)pos * half + (c < half ? c : c - half)) * 2);
                cs[h] = t2.x;
                sn[h] = t2.y;
            }
        }
    }
    if (live) {
#pragma unroll
        for (int h = 0; h < DH; h++) {
            float p = pv[h][0];
#pragma unroll
            for (int s = 1; s < SU; s++) p = p + pv[h][s];
            for (int s = SU; s < splits; s++) p = p + part[((size_t)s * M + m) * N + hidx * D + 64 * h + lane];
            buf[wave][64 * h + lane] = p * f;
        }
    }
    __syncthreads();
    // q_norm / k_norm (model.js:388-394): rmsnorm over the head's D values
    // (lane partials, then a wave reduction), before RoPE reads neighbouring
    // channels
    if (ex.qn) {   // a kernel argument: the barrier is uniform
        if (live && hidx < nH + nKV) {
            const float* w = hidx < nH ? ex.qn : ex.kn;
            float ss = 0.0f;
            for (int d = lane; d < D; d += 64) ss += buf[wave][d] * buf[wave][d];
            ss = wave_sum(ss);
            const float scale = 1.0f / sqrtf(ss / (float)D + ex.eps);
            for (int d = lane; d < D; d += 64) buf[wave][d] = buf[wave][d] * scale * w[d];
        }
        __syncthreads();
    }
    if (live && hidx < nH) {
        if (do_q) {
#pragma unroll
            for (int h = 0; h < DH; h++) rq[wave][64 * h + lane] = rope_cs(buf[wave], 64 * h + lane, rot, cs[h], sn[h]);
        }
    }
    __syncthreads();
    if (!live) return;
    if (hidx >= nqkv) {
        // the output gate's raw values (times the row factor), for the combine
        if (do_q) {
            float* gr = ex.gate + (size_t)m * nH * D + (size_t)(hidx - nqkv) * D;
            for (int d = lane; d < D; d += 64) gr[d] = buf[wave][d];
        }
        return;
    }
    if (hidx < nH) {
        if (!do_q) return;
        if (lane < D / 8) {
            const int d0 = 8 * lane;
            half8_t hi, lo;
            // the lane's 8 channels as two 16-byte reads
            const float4 qa = *(const float4*)&rq[wave][d0], qb = *(const float4*)&rq[wave][d0 + 4];
            const float qv[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
#pragma unroll
            for (int j = 0; j < 8; j++) {
                _Float16 a, b;
                split_hilo(qv[j], a, b);
                hi[j] = a;
                lo[j] = b;
            }
            const int kvh = hidx / group, gi = hidx % group;
            const int rho = i * group + gi;
            const int mtq = rho >> 4, ln = (rho & 15) + 16 * ((d0 & 31) >> 3), grp = d0 >> 5;
            const size_t at = (size_t)jb.qp_off + ((((size_t)kvh * jb.mtq + mtq) * g.ng + grp) * 2) * 64 + ln;
            Qp[at] = __builtin_bit_cast(uint4, hi);
            Qp[at + 64] = __builtin_bit_cast(uint4, lo);
        }
        return;
    }
    if (!do_kv) return;
    const int which = hidx < nH + nKV ? 0 : 1;
    const int n = hidx - nH - which * nKV;
    const int s = pos % g.page;
    uint8_t* blk = (which ? vpool : kpool) + ((size_t)page * nKV + n) * g.blk;
#pragma unroll
    for (int h = 0; h < DH; h++) {
        const int d = 64 * h + lane;
        const float v = which ? buf[wave][d] : rope_cs(buf[wave], d, rot, cs[h], sn[h]);
        float amax = fabsf(v);
        for (int o = 1; o < 32; o <<= 1) amax = fmaxf(amax, __shfl_xor(amax, o));
        const float scale = amax / 127.0f;
        const float inv = scale > 0.0f ? 1.0f / scale : 0.0f;
        float q = __builtin_rintf(v * inv);
        q = fminf(fmaxf(q, -127.0f), 127.0f);
        const int8_t code = (int8_t)(int)q;
        const int b = d >> 5;
        if (which == 0) {
            blk[(size_t)s * D + kpos(d, D)] = (uint8_t)((uint8_t)code ^ 0x80u);
            if ((d & 31) == 0) *(float*)(blk + 64 * D + ((size_t)s * g.ng + b) * 4) = scale;
        } else {
            blk[vcode_at(d, s, D)] = (uint8_t)((uint8_t)code ^ 0x80u);
            if ((d & 31) == 0) *(float*)(blk + 64 * D + (size_t)vscale_at(b, s, g.ng) * 4) = scale;
        }
    }
}

template <int D>
static void launch_fin_qkv_d(hipStream_t st, dim3 grid, const float* part, int splits, int M, const int32_t* row_job,
                             const JobDev* jobs, int nH, int group, const KVGeom& g, const float* tbl, int rot,
                             uint8_t* kpool, uint8_t* vpool, const uint32_t* page_table, uint4* Qp,
                             const RowScale& rs, int do_q, int do_kv, const QkExtras& ex) {
    if (splits <= 4)
        hipLaunchKernelGGL((k_fin_qkv<D, 4>), grid, dim3(256), 0, st, part, splits, M, row_job, jobs, nH, group, g,
                           tbl, rot, kpool, vpool, page_table, Qp, rs, do_q, do_kv, ex);
    else
        hipLaunchKernelGGL((k_fin_qkv<D, 16>), grid, dim3(256), 0, st, part, splits, M, row_job, jobs, nH, group, g,
                           tbl, rot, kpool, vpool, page_table, Qp, rs, do_q, do_kv, ex);
}

void launch_fin_qkv(hipStream_t st, const float* part, int splits, int M, const int32_t* row_job,
                    const JobDev* jobs, int nH, int group, const KVGeom& g, const float* tbl, int rot,
                    uint8_t* kpool, uint8_t* vpool, const uint32_t* page_table, uint4* Qp, const RowScale& rs,
                    int do_q, int do_kv, const QkExtras& ex) {
    const int nall = nH + 2 * g.nKV + (ex.gate ? nH : 0);
    const dim3 grid((nall + 3) / 4, M);
    if (g.D == 256)
        launch_fin_qkv_d<256>(st, grid, part, splits, M, row_job, jobs, nH, group, g, tbl, rot, kpool, vpool,
                              page_table, Qp, rs, do_q, do_kv, ex);
    else if (g.D == 128)
        launch_fin_qkv_d<128>(st, grid, part, splits, M, row_job, jobs, nH, group, g, tbl, rot, kpool, vpool,
                              page_table, Qp, rs, do_q, do_kv, ex);
    else
        launch_fin_qkv_d<64>(st, grid, part, splits, M, row_job, jobs, nH, group, g, tbl, rot, kpool, vpool,
                             page_table, Qp, rs, do_q, do_kv, ex);
    CHECK_LAUNCH();
}

// =========================================================== Gated DeltaNet ===
// A hybrid checkpoint's linear_attention blocks (web/model/model.js:418-527,
// web/model/kernels.js:1531-1839) over the packed jobs, each on its own
// session's state. Three kernels after the fused in_proj matmul:
//   k_lin_conv  planes summed (times the input rmsnorm's row factor), the
//               depthwise causal conv + SiLU through the job's rows with the
//               session's ring, the ring advanced; z, b, a passed through;
//   k_gdn       the gated delta rule with the q/k l2norm folded in;
//   k_lin_norm  RMSNormGated times silu(z) into the out_proj operand.

// Plane sum of one column in plane order, times the row factor.
__device__ static inline float plane_col(const float* part, int splits, int M, int N, int m, int col, float f) {
    float p = part[(size_t)m * N + col];
    for (int s = 1; s < splits; s++) p = p + part[((size_t)s * M + m) * N + col];
    return p * f;
}

// causal_conv1d (kernels.js:1538-1580) + update_conv_history (:1582-1620).
// One thread per (job, channel) walks the job's rows in order, so the ring
// (the K-1 raw rows before the current one) stays in registers: it is read
// from the session's state first (zeros for a job at position 0, a new
// session) and written back after the job's last row. Per row: acc = sum over
// k of w[c][k] * x[t-(K-1)+k] in k order, out = acc * (1/(1+exp(-acc))).
// Speculation (model.js:447-470): a rollback job starts from the snapshot's
// ring, advances it through the kept rows' stored raw values and copies
// their stored outputs (and b, a) to `lrep` for the recurrence; a verify
// writes the ring it starts from to the snapshot and stores each row's raw
// value and output. The thread that reads a stored row is the one that
// overwrites it, so a rollback job that is also a verify is ordered.
__global__ __launch_bounds__(256) void k_lin_conv(const float* __restrict__ part, int splits, int M,
                                                  const JobDev* __restrict__ jobs, RowScale rs,
                                                  const float* __restrict__ conv, LinGeom lg,
                                                  float* __restrict__ state, float* __restrict__ lraw,
                                                  float* __restrict__ lrep) {
    constexpr int K = LIN_CONV_K;
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= lg.W) return;
    const int j = blockIdx.y;
    const JobDev jb = jobs[j];
    float* base = state + (size_t)jb.slot * lg.sstride;
    float* rep = base + lg.rep_off;
    float* lr = lrep + (size_t)j * LIN_SPEC_ROWS * lg.lrep_w;
    const int keep = jb.keep > 0 ? jb.keep : 0;
    // plane column: q|k|v|z in place, b and a each padded to nVp rows
    const int col = c < lg.convDim + lg.valueDim + lg.nV ? c : c - lg.nV + lg.nVp;
    if (c >= lg.convDim) {
        // z, b, a pass through; b and a also feed a rollback's and a verify's rows
        const bool ba = c >= lg.convDim + lg.valueDim;
        const int e = c - lg.convDim - lg.valueDim;   // b: [0, nV), a: [nV, 2nV)
        if (ba)
            for (int i = 0; i < keep; i++)
                lr[(size_t)i * lg.lrep_w + lg.convDim + e] = rep[(size_t)i * lg.rep_w + 2 * lg.convDim + e];
        for (int i = 0; i < jb.n; i++) {
            const int m = jb.row0 + i;
            const float v = plane_col(part, splits, M, lg.N, m, col, row_scale(rs, m));
            lraw[(size_t)m * lg.W + c] = v;
            if (ba && jb.snap) rep[(size_t)i * lg.rep_w + 2 * lg.convDim + e] = v;
        }
        return;
    }
    float* cur = base + lg.hist_off + c;            // [K-1][convDim]
    float* snap = base + lg.blk + lg.hist_off + c;
    const float* src = jb.keep >= 0 ? snap : cur;
    float h[K - 1];
#pragma unroll
    for (int r = 0; r < K - 1; r++) h[r] = jb.past > 0 ? src[(size_t)r * lg.convDim] : 0.0f;
    for (int i = 0; i < keep; i++) {
        lr[(size_t)i * lg.lrep_w + c] = rep[(size_t)i * lg.rep_w + lg.convDim + c];
#pragma unroll
        for (int k = 0; k < K - 2; k++) h[k] = h[k + 1];
        h[K - 2] = rep[(size_t)i * lg.rep_w + c];
    }
    if (jb.snap) {
#pragma unroll
        for (int r = 0; r < K - 1; r++) snap[(size_t)r * lg.convDim] = h[r];
    }
    float w[K];
#pragma unroll
    for (int k = 0; k < K; k++) w[k] = conv[(size_t)c * K + k];
    for (int i = 0; i < jb.n; i++) {
        const int m = jb.row0 + i;
        const float x = plane_col(part, splits, M, lg.N, m, col, row_scale(rs, m));
        float acc = 0.0f;
#pragma unroll
        for (int k = 0; k < K - 1; k++) acc = acc + w[k] * h[k];
        acc = acc + w[K - 1] * x;
        const float sg = 1.0f / (1.0f + expf(-acc));
        const float out = acc * sg;
        lraw[(size_t)m * lg.W + c] = out;
        if (jb.snap) {
            rep[(size_t)i * lg.rep_w + c] = x;
            rep[(size_t)i * lg.rep_w + lg.convDim + c] = out;
        }
#pragma unroll
        for (int k = 0; k < K - 2; k++) h[k] = h[k + 1];
        h[K - 2] = x;
    }
#pragma unroll
    for (int r = 0; r < K - 1; r++) cur[(size_t)r * lg.convDim] = h[r];
}

void launch_lin_conv(hipStream_t st, const float* part, int splits, int M, int njobs, const JobDev* jobs,
                     const RowScale& rs, const float* conv, const LinGeom& lg, float* state, float* lraw,
                     float* lrep) {
    if (njobs <= 0) return;
    hipLaunchKernelGGL(k_lin_conv, dim3((lg.W + 255) / 256, njobs), dim3(256), 0, st, part, splits, M, jobs, rs,
                       conv, lg, state, lraw, lrep);
    CHECK_LAUNCH();
}

// The same conv for a pass with a long job (a prefill chunk), parallel over
// rows, in three steps (the arithmetic per row is the one above, so the bits
// do not depend on the path):
//   k_lin_ring_pre   the ring each job starts from (the session's, or the
//                    snapshot's advanced through the kept rows) into `lring`
//                    [job][K-1][convDim]; the rollback rows to `lrep`; a
//                    verify's snapshot ring;
//   k_lin_conv_rows  one thread per (row, channel): the window from the
//                    job's own rows (planes summed again) and `lring`;
//   k_lin_ring_post  the ring after the job's last row, into the session.
__global__ __launch_bounds__(256) void k_lin_ring_pre(const JobDev* __restrict__ jobs, LinGeom lg,
                                                      float* __restrict__ state, float* __restrict__ lrep,
                                                      float* __restrict__ lring) {
    constexpr int K = LIN_CONV_K;
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= lg.W) return;
    const int j = blockIdx.y;
    const JobDev jb = jobs[j];
    float* base = state + (size_t)jb.slot * lg.sstride;
    const float* rep = base + lg.rep_off;
    float* lr = lrep + (size_t)j * LIN_SPEC_ROWS * lg.lrep_w;
    const int keep = jb.keep > 0 ? jb.keep : 0;
    if (c >= lg.convDim) {
        if (c >= lg.convDim + lg.valueDim) {
            const int e = c - lg.convDim - lg.valueDim;
            for (int i = 0; i < keep; i++)
                lr[(size_t)i * lg.lrep_w + lg.convDim + e] = rep[(size_t)i * lg.rep_w + 2 * lg.convDim + e];
        }
        return;
    }
    float* cur = base + lg.hist_off + c;
    float* snap = base + lg.blk + lg.hist_off + c;
    const float* src = jb.keep >= 0 ? snap : cur;
    float h[K - 1];
#pragma unroll
    for (int r = 0; r < K - 1; r++) h[r] = jb.past > 0 ? src[(size_t)r * lg.convDim] : 0.0f;
    for (int i = 0; i < keep; i++) {
        lr[(size_t)i * lg.lrep_w + c] = rep[(size_t)i * lg.rep_w + lg.convDim + c];
#pragma unroll
        for (int k = 0; k < K - 2; k++) h[k] = h[k + 1];
        h[K - 2] = rep[(size_t)i * lg.rep_w + c];
    }
    float* e = lring + (size_t)j * (K - 1) * lg.convDim + c;
#pragma unroll
    for (int r = 0; r < K - 1; r++) {
        e[(size_t)r * lg.convDim] = h[r];
        if (jb.snap) snap[(size_t)r * lg.convDim] = h[r];
    }
}

__global__ __launch_bounds__(256) void k_lin_conv_rows(const float* __restrict__ part, int splits, int M,
                                                       const int32_t* __restrict__ row_job,
                                                       const JobDev* __restrict__ jobs, RowScale rs,
                                                       const float* __restrict__ conv, LinGeom lg,
                                                       float* __restrict__ state, const float* __restrict__ lring,
                                                       float* __restrict__ lraw) {
    constexpr int K = LIN_CONV_K;
    const int c = blockIdx.x * 256 + threadIdx.x;
    const int m = blockIdx.y;
    if (c >= lg.W || m >= M) return;
    const int j = row_job[m];
    const JobDev jb = jobs[j];
    const int i = m - jb.row0;
    float* rep = state + (size_t)jb.slot * lg.sstride + lg.rep_off;
    const int col = c < lg.convDim + lg.valueDim + lg.nV ? c : c - lg.nV + lg.nVp;
    if (c >= lg.convDim) {
        const float v = plane_col(part, splits, M, lg.N, m, col, row_scale(rs, m));
        lraw[(size_t)m * lg.W + c] = v;
        if (jb.snap && c >= lg.convDim + lg.valueDim) rep[(size_t)i * lg.rep_w + 2 * lg.convDim + (c - lg.convDim - lg.valueDim)] = v;
        return;
    }
    const float* e = lring + (size_t)j * (K - 1) * lg.convDim + c;
    float x[K];   // the window: rows i-K+1 .. i
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int t = i - (K - 1) + k;
        x[k] = t >= 0 ? plane_col(part, splits, M, lg.N, jb.row0 + t, col, row_scale(rs, jb.row0 + t))
                      : e[(size_t)(K - 1 + t) * lg.convDim];
    }
    float acc = 0.0f;
#pragma unroll
    for (int k = 0; k < K; k++) acc = acc + conv[(size_t)c * K + k] * x[k];
    const float sg = 1.0f / (1.0f + expf(-acc));
    const float out = acc * sg;
    lraw[(size_t)m * lg.W + c] = out;
    if (jb.snap) {
        rep[(size_t)i * lg.rep_w + c] = x[K - 1];
        rep[(size_t)i * lg.rep_w + lg.convDim + c] = out;
    }
}

__global__ __launch_bounds__(256) void k_lin_ring_post(const float* __restrict__ part, int splits, int M,
                                                       const JobDev* __restrict__ jobs, RowScale rs, LinGeom lg,
                                                       float* __restrict__ state, const float* __restrict__ lring) {
    constexpr int K = LIN_CONV_K;
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= lg.convDim) return;
    const int j = blockIdx.y;
    const JobDev jb = jobs[j];
    float* cur = state + (size_t)jb.slot * lg.sstride + lg.hist_off + c;
    const float* e = lring + (size_t)j * (K - 1) * lg.convDim + c;
#pragma unroll
    for (int r = 0; r < K - 1; r++) {
        const int t = jb.n - (K - 1) + r;   // the ring's row r after the job
        cur[(size_t)r * lg.convDim] = t >= 0 ? plane_col(part, splits, M, lg.N, jb.row0 + t, c, row_scale(rs, jb.row0 + t))
                                             : e[(size_t)(K - 1 + t) * lg.convDim];
    }
}

void launch_lin_conv_rows(hipStream_t st, const float* part, int splits, int M, int njobs, const int32_t* row_job,
                          const JobDev* jobs, const RowScale& rs, const float* conv, const LinGeom& lg, float* state,
                          float* lraw, float* lrep, float* lring) {
    if (njobs <= 0 || M <= 0) return;
    const int bw = (lg.W + 255) / 256;
    hipLaunchKernelGGL(k_lin_ring_pre, dim3(bw, njobs), dim3(256), 0, st, jobs, lg, state, lrep, lring);
    hipLaunchKernelGGL(k_lin_conv_rows, dim3(bw, M), dim3(256), 0, st, part, splits, M, row_job, jobs, rs, conv, lg,
                       state, lring, lraw);
    hipLaunchKernelGGL(k_lin_ring_post, dim3((lg.convDim + 255) / 256, njobs), dim3(256), 0, st, part, splits, M, jobs,
                       rs, lg, state, lring);
    CHECK_LAUNCH();
}

// gated_delta_net_step (kernels.js:1672-1805) for every row of a job, on its
// session's S [nV][Dk][Dv]. Per token, with the l2norm of the head's q and k
// (l2norm_heads, kernels.js:1622-1670; source head h / group, the value-head
// repeat) folded in as k^ = k/sqrt(sum k^2 + 1e-6) and q^ likewise, times
// 1/sqrt(Dk):
//   g = exp(-exp(A_log) * softplus(a + dt_bias)), beta = sigmoid(b);
//   delta = (v - g*(s.k^)) * beta; out = g*(s.q^) + delta*(k^.q^);
//   s = g*s + k^*delta.
// A job at position 0 starts from a zero state. A rollback job starts from
// the snapshot and first re-runs the kept rows (from `lrep`, no output); a
// verify writes the state it starts from to the snapshot.
//
// A workgroup serves (32 value columns, value head, job), eight threads a
// column with DK/8 rows of it each, in registers for the whole job. Two
// kernels, the same operations on the same operands in the same order, so a
// row's bits depend on neither its job's length nor its batch-mates:
//   k_gdn_few  jobs of few rows (gdn_takes_few): bound by the state's
//              read and write, so few registers (many workgroups to hide the
//              reads), whole 128-byte rows of state a load, the columns' sums
//              through LDS with a barrier a token;
//   k_gdn      longer jobs: bound by the chain from token to token, so a
//              column's eight threads are neighbouring lanes and its sums DPP
//              adds with no barrier, and what a token needs that does not
//              depend on the state (k^, q^, k^.q^, g, beta, the columns' v) is
//              formed GDN_CH tokens at a time, a token a wave, and read
//              from LDS a token ahead; the next tokens' inputs load under the
//              walk.
// A single kernel that formed the dot products of q and k beside the state's
// and read each token's inputs as it came to them took 1.49 us a row of a
// long job: 512 rows 759 us a block (48 heads of 128 x 128), now 203.
constexpr int GDN_TV = 32, GDN_T = 256, GDN_CH = 16, GDN_KG = 8;
static_assert(LIN_SPEC_ROWS < GDN_CH, "a rollback's kept rows and the row after them fall in one chunk");
// Sum over the eight lanes 8i .. 8i+7, in all of them:
// ((x0 + x1) + (x2 + x3)) + ((x4 + x5) + (x6 + x7)).
__device__ static inline float sum8(float x) {
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0xB1, 0xf, 0xf, true));   // lane ^ 1
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x4E, 0xf, 0xf, true));   // lane ^ 2
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x141, 0xf, 0xf, true));  // 7 - lane of the eight
    return x;
}
// A token's inputs across a wave: q and k of the head, lane l holding
// channels l and l + 64, and their sums of squares and product.
template <int DK>
struct GdnRow {
    static constexpr int PER = (DK + 63) / 64;
    float q[PER], k[PER];
};
template <int DK>
__device__ static inline void gdn_load(GdnRow<DK>& x, const float* row, int keyDim, int kh, int lane) {
#pragma unroll
    for (int e = 0; e < GdnRow<DK>::PER; e++) {
        const int d = lane + 64 * e;
        x.q[e] = d < DK ? row[kh * DK + d] : 0.0f;
        x.k[e] = d < DK ? row[keyDim + kh * DK + d] : 0.0f;
    }
}
// q.q, k.k and k.q of T tokens, their sums across the wave side by side.
template <int DK, int T>
__device__ static inline void gdn_norms(const GdnRow<DK> (&x)[T], float (&n3)[T][3]) {
#pragma unroll
    for (int t = 0; t < T; t++) {
        n3[t][0] = n3[t][1] = n3[t][2] = 0.0f;
#pragma unroll
        for (int e = 0; e < GdnRow<DK>::PER; e++) {
            n3[t][0] = __builtin_fmaf(x[t].q[e], x[t].q[e], n3[t][0]);
            n3[t][1] = __builtin_fmaf(x[t].k[e], x[t].k[e], n3[t][1]);
            n3[t][2] = __builtin_fmaf(x[t].k[e], x[t].q[e], n3[t][2]);
        }
    }
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int i = 0; i < 3; i++) n3[t][i] = sum8(n3[t][i]);
#pragma unroll
    for (int o = 8; o < 64; o <<= 1)
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int i = 0; i < 3; i++) n3[t][i] += __shfl_xor(n3[t][i], o);
}
// The factors of q and k, from their sums: q's carries 1/sqrt(Dk).
struct GdnScale {
    float rq, rk, kq, g, beta;
};
__device__ static inline GdnScale gdn_scale(const float (&n3)[3], float q_scale, float A, float dtb, float a, float b) {
    GdnScale r;
    r.rq = q_scale / sqrtf(n3[0] + 1e-6f);
    r.rk = 1.0f / sqrtf(n3[1] + 1e-6f);
    r.kq = n3[2] * r.rq * r.rk;
    const float x = a + dtb;
    const float sp = x > 20.0f ? x + logf(1.0f + expf(-x)) : logf(1.0f + expf(x));
    r.g = expf(-A * sp);
    r.beta = 1.0f / (1.0f + expf(-b));
    return r;
}

template <int DK>
__global__ __launch_bounds__(GDN_T) void k_gdn_few(const float* __restrict__ lraw, const float* __restrict__ lrep,
                                                   const JobDev* __restrict__ jobs, const float* __restrict__ gp,
                                                   LinGeom lg, float* __restrict__ state, float* __restrict__ core) {
    constexpr int ROWS = DK / GDN_KG;
    __shared__ float pkv[2][GDN_KG][GDN_TV], pqo[2][GDN_KG][GDN_TV];
    const int h = blockIdx.y, j = blockIdx.z;
    const JobDev jb = jobs[j];
    const int lane = threadIdx.x & 63, col = threadIdx.x % GDN_TV, kg = threadIdx.x / GDN_TV;
    const int vv = blockIdx.x * GDN_TV + col;
    const bool live = vv < lg.Dv;
    const int vvc = live ? vv : lg.Dv - 1;   // out-of-range columns read a real one and discard it
    const int k0 = kg * ROWS, kh = h / lg.group;
    float* S = state + (size_t)jb.slot * lg.sstride + (size_t)h * DK * lg.Dv;   // current
    float* Ssnap = S + lg.blk;                                                   // snapshot
    const float* src = jb.keep >= 0 ? Ssnap : S;
    float s[ROWS];
#pragma unroll
    for (int i = 0; i < ROWS; i++) s[i] = (jb.past > 0 && live) ? src[(size_t)(k0 + i) * lg.Dv + vv] : 0.0f;
    const float A = expf(gp[h]), dtb = gp[lg.nV + h];
    const float q_scale = 1.0f / sqrtf((float)DK);
    const int keep = jb.keep > 0 ? jb.keep : 0, total = keep + jb.n;   // the kept rows first, then the job's
    const float* lr = lrep + (size_t)j * LIN_SPEC_ROWS * lg.lrep_w;
    for (int t = 0; t < total; t++) {
        const int i = t - keep;   // the job's row, < 0: a kept one
        const float* row = i < 0 ? lr + (size_t)t * lg.lrep_w : lraw + (size_t)(jb.row0 + i) * lg.W;
        const int boff = i < 0 ? lg.convDim : lg.convDim + lg.valueDim;
        GdnRow<DK> x[1];
        gdn_load<DK>(x[0], row, lg.keyDim, kh, lane);
        float kx[ROWS], qx[ROWS];
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            qx[r] = row[kh * DK + k0 + r];
            kx[r] = row[lg.keyDim + kh * DK + k0 + r];
        }
        const float v = row[2 * lg.keyDim + h * lg.Dv + vvc], b = row[boff + h], a = row[boff + lg.nV + h];
        if (i == 0 && jb.snap && live) {
#pragma unroll
            for (int r = 0; r < ROWS; r++) Ssnap[(size_t)(k0 + r) * lg.Dv + vv] = s[r];
        }
        float n3[1][3];
        gdn_norms<DK, 1>(x, n3);
        const GdnScale sc = gdn_scale(n3[0], q_scale, A, dtb, a, b);
        float kv[2] = {0.0f, 0.0f}, qo[2] = {0.0f, 0.0f};   // even and odd rows
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            kx[r] = kx[r] * sc.rk;
            kv[r & 1] = __builtin_fmaf(s[r], kx[r], kv[r & 1]);
            qo[r & 1] = __builtin_fmaf(s[r], qx[r] * sc.rq, qo[r & 1]);
        }
        const int buf = t & 1;
        pkv[buf][kg][col] = kv[0] + kv[1];
        pqo[buf][kg][col] = qo[0] + qo[1];
        __syncthreads();
        auto tree = [&](const float (&p)[GDN_KG][GDN_TV]) {   // sum8's order
            return ((p[0][col] + p[1][col]) + (p[2][col] + p[3][col])) +
                   ((p[4][col] + p[5][col]) + (p[6][col] + p[7][col]));
        };
        const float kvT = tree(pkv[buf]);
        const float delta = (v - sc.g * kvT) * sc.beta;
#pragma unroll
        for (int r = 0; r < ROWS; r++) s[r] = __builtin_fmaf(sc.g, s[r], kx[r] * delta);
        if (i >= 0 && kg == 0 && live)
            core[(size_t)(jb.row0 + i) * lg.valueDim + h * lg.Dv + vv] =
                __builtin_fmaf(sc.g, tree(pqo[buf]), delta * sc.kq);
    }
    if (live) {
#pragma unroll
        for (int i = 0; i < ROWS; i++) S[(size_t)(k0 + i) * lg.Dv + vv] = s[i];
    }
}

template <int DK>
__global__ __launch_bounds__(GDN_T, 3) void k_gdn(const float* __restrict__ lraw, const float* __restrict__ lrep,
                                                  const JobDev* __restrict__ jobs, const float* __restrict__ gp,
                                                  LinGeom lg, float* __restrict__ state, float* __restrict__ core) {
    // a lane group's ROWS values start 4 floats further than the last group's
    // end at DK = 128, so the eight groups' 16-byte reads fall in different banks
    constexpr int ROWS = DK / GDN_KG, LROW = ROWS == 16 ? 20 : ROWS, LK = LROW * GDN_KG;
    constexpr int TPW = GDN_CH / (GDN_T / 64);   // tokens a wave
    __shared__ __align__(16) float s_k[GDN_CH][LK], s_q[GDN_CH][LK], s_v[GDN_CH][GDN_TV];
    __shared__ __align__(16) float s_sc[GDN_CH][4];   // g, beta, k^.q^
    const int h = blockIdx.y, j = blockIdx.z;
    const JobDev jb = jobs[j];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = lane & 7, cw = wave * 8 + (lane >> 3);
    const int vv = blockIdx.x * GDN_TV + cw;
    const bool live = vv < lg.Dv;
    const int k0 = kg * ROWS, kh = h / lg.group;
    float* S = state + (size_t)jb.slot * lg.sstride + (size_t)h * DK * lg.Dv;   // current
    float* Ssnap = S + lg.blk;                                                   // snapshot
    // the lane's elements through one offset register (a lane past Dv reads and
    // writes past the resource's end: zero, dropped)
    const int sb = DK * lg.Dv * 4, so = live ? (k0 * lg.Dv + vv) * 4 : sb;
    float s[ROWS];
    {
        const auto r = __builtin_amdgcn_make_buffer_rsrc((void*)(jb.keep >= 0 ? Ssnap : S), 0, jb.past > 0 ? sb : 0,
                                                         0x00020000);
#pragma unroll
        for (int i = 0; i < ROWS; i++)
            s[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, so, i * lg.Dv * 4, 0));
    }
    auto put_state = [&](float* to) {
        const auto r = __builtin_amdgcn_make_buffer_rsrc((void*)to, 0, sb, 0x00020000);
#pragma unroll
        for (int i = 0; i < ROWS; i++)
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(s[i]), r, so, i * lg.Dv * 4, 0);
    };
    const float A = expf(gp[h]), dtb = gp[lg.nV + h];
    const float q_scale = 1.0f / sqrtf((float)DK);
    const int keep = jb.keep > 0 ? jb.keep : 0, total = keep + jb.n;   // the kept rows first, then the job's
    const float* lr = lrep + (size_t)j * LIN_SPEC_ROWS * lg.lrep_w;
    // this wave's tokens of the chunk at t0: wave, wave + 4, ...
    GdnRow<DK> x[TPW];
    float vr[TPW], ar[TPW], br[TPW];
    auto load = [&](int t0) {
#pragma unroll
        for (int u = 0; u < TPW; u++) {
            const int i = min(t0 + wave + u * (GDN_T / 64), total - 1);   // past the end: loaded and not used
            const float* row = i < keep ? lr + (size_t)i * lg.lrep_w : lraw + (size_t)(jb.row0 + i - keep) * lg.W;
            const int boff = i < keep ? lg.convDim : lg.convDim + lg.valueDim;
            gdn_load<DK>(x[u], row, lg.keyDim, kh, lane);
            const int c = blockIdx.x * GDN_TV + (lane & (GDN_TV - 1));
            vr[u] = row[2 * lg.keyDim + h * lg.Dv + (c < lg.Dv ? c : lg.Dv - 1)];
            br[u] = row[boff + h];
            ar[u] = row[boff + lg.nV + h];
        }
    };
    auto prepare = [&](int t0) {
        float n3[TPW][3];
        gdn_norms<DK, TPW>(x, n3);
#pragma unroll
        for (int u = 0; u < TPW; u++) {
            const int c = wave + u * (GDN_T / 64);
            if (t0 + c >= total) continue;
            const GdnScale sc = gdn_scale(n3[u], q_scale, A, dtb, ar[u], br[u]);
#pragma unroll
            for (int e = 0; e < GdnRow<DK>::PER; e++) {
                const int d = lane + 64 * e;
                if (d < DK) {
                    const int at = (d / ROWS) * LROW + d % ROWS;
                    s_q[c][at] = x[u].q[e] * sc.rq;
                    s_k[c][at] = x[u].k[e] * sc.rk;
                }
            }
            if (lane < GDN_TV) s_v[c][lane] = vr[u];
            if (lane == 0) *(float4*)s_sc[c] = make_float4(sc.g, sc.beta, sc.kq, 0.0f);
        }
    };
    struct Tok {
        float k[ROWS], q[ROWS], v;
        float4 sc;
    };
    auto fetch = [&](Tok& y, int c) {
        if constexpr (ROWS >= 4) {
#pragma unroll
            for (int r = 0; r < ROWS; r += 4) {
                const float4 ka = *(const float4*)&s_k[c][kg * LROW + r], qa = *(const float4*)&s_q[c][kg * LROW + r];
                y.k[r] = ka.x; y.k[r + 1] = ka.y; y.k[r + 2] = ka.z; y.k[r + 3] = ka.w;
                y.q[r] = qa.x; y.q[r + 1] = qa.y; y.q[r + 2] = qa.z; y.q[r + 3] = qa.w;
            }
        } else {
#pragma unroll
            for (int r = 0; r < ROWS; r++) {
                y.k[r] = s_k[c][kg * LROW + r];
                y.q[r] = s_q[c][kg * LROW + r];
            }
        }
        y.sc = *(const float4*)s_sc[c];
        y.v = s_v[c][cw];
    };
    auto advance = [&](const Tok& y, float* o) {
        float kv[2] = {0.0f, 0.0f}, qo[2] = {0.0f, 0.0f};   // even and odd rows
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            kv[r & 1] = __builtin_fmaf(s[r], y.k[r], kv[r & 1]);
            qo[r & 1] = __builtin_fmaf(s[r], y.q[r], qo[r & 1]);
        }
        const float kvT = sum8(kv[0] + kv[1]), qoT = sum8(qo[0] + qo[1]);
        const float delta = (y.v - y.sc.x * kvT) * y.sc.y;
#pragma unroll
        for (int r = 0; r < ROWS; r++) s[r] = __builtin_fmaf(y.sc.x, s[r], y.k[r] * delta);
        if (o && kg == 0 && live) *o = __builtin_fmaf(y.sc.x, qoT, delta * y.sc.z);
    };
    // tokens c0 .. c1-1 of the chunk; `o`: their outputs, a row apart
    auto walk = [&](int c0, int c1, float* o) {
        if (c0 >= c1) return;
        const size_t os = o ? lg.valueDim : 0;
        Tok y, z;
        fetch(y, c0);
        int c = c0;
        for (; c + 2 <= c1; c += 2) {
            fetch(z, c + 1);
            __builtin_amdgcn_sched_barrier(0);
            advance(y, o);
            fetch(y, min(c + 2, GDN_CH - 1));   // past the last token: read and not used
            __builtin_amdgcn_sched_barrier(0);
            advance(z, o ? o + os : nullptr);
            o += 2 * os;
        }
        if (c < c1) advance(y, o);
    };
    load(0);
    for (int t0 = 0; t0 < total; t0 += GDN_CH) {
        prepare(t0);
        __syncthreads();
        if (t0 + GDN_CH < total) load(t0 + GDN_CH);   // in flight under the walk
        const int nt = min(GDN_CH, total - t0);
        int c0 = 0;
        if (t0 == 0) {   // the kept rows are all in the first chunk
            c0 = keep;
            walk(0, c0, nullptr);
            if (jb.snap) put_state(Ssnap);
        }
        walk(c0, nt, core + (size_t)(jb.row0 + t0 + c0 - keep) * lg.valueDim + h * lg.Dv + vv);
        __syncthreads();   // the chunk's LDS is free
    }
    put_state(S);
}

// Which kernel a launch takes, from the rows its jobs walk (a rollback's kept
// rows among them), their sum over the jobs and the longest job's, and the
// verifies, which write the state twice. With many workgroups a CU the work
// decides: k_gdn_few takes about 0.95 us a job and 0.37 a verify less than
// k_gdn and 0.28 us a row more (48 heads of 128 x 128), so the line is three
// rows a job on average, and a fourth for a verify. With few the longest
// job's chain does, 0.9 us a row longer in k_gdn_few, against a start of k_gdn
// that grows with the workgroups.
// Launches of 48 heads of 128 x 128, k_gdn_few / k_gdn, us (16, 4 and 1 jobs):
//   1 row 22.7/33.5, 7.0/9.2, 4.9/5.6         2 rows 28.1/35.2, 9.1/10.3, 5.5/6.1
//   3 rows (2 of them kept) 34.1/36.0, 11.3/10.6, 6.6/6.2
//   4 rows 40.0/38.0, 12.6/11.2, 7.8/6.8      8 rows 63.4/43.0, 20.7/14.2, 12.7/7.9
//   verifies of 4 rows 46.7/50.5, 13.9/13.9, 8.6/7.5, of 5 51.9/51.0, 16.0/14.4, 9.9/8.2
//   1 row after 8 kept ones 68.8/42.1, 22.2/13.3, 13.2/7.8
//   5 rows beside 15 (3) jobs of one 24.3/33.8 (11.3/10.7), 17 beside 15 30.4/35.7, 32 beside 15 47.1/36.2
// Over 426 mixes of 1-16 jobs of 1-48 rows (this shape, 16 heads of it, 32
// heads of 64 x 64) the rule's choice takes 0.2% more than the better kernel
// on average and 17% (1.4 us) at worst; a line on the longest job's new rows
// alone (4) took 8% more on average and up to 94%.
static bool gdn_takes_few(int njobs, const GdnRows& r, const LinGeom& lg, int ncu) {
    const long long groups = (long long)njobs * lg.nV * ((lg.Dv + GDN_TV - 1) / GDN_TV);
    return r.walked <= 3 * njobs + r.verifies && r.longest <= std::max(2LL, 2 * groups / ncu - 5);
}

template <int DK>
static void launch_gdn_dk(hipStream_t st, const float* lraw, const float* lrep, int njobs, const JobDev* jobs,
                          const float* gp, const LinGeom& lg, float* state, float* core, bool few) {
    const dim3 grid((lg.Dv + GDN_TV - 1) / GDN_TV, lg.nV, njobs), blk(GDN_T);
    if (few)
        hipLaunchKernelGGL(k_gdn_few<DK>, grid, blk, 0, st, lraw, lrep, jobs, gp, lg, state, core);
    else
        hipLaunchKernelGGL(k_gdn<DK>, grid, blk, 0, st, lraw, lrep, jobs, gp, lg, state, core);
}

void launch_gdn(hipStream_t st, const float* lraw, const float* lrep, int njobs, const JobDev* jobs, const float* gp,
                const LinGeom& lg, float* state, float* core, const GdnRows& rows, int ncu) {
    if (njobs <= 0) return;
    const bool few = gdn_takes_few(njobs, rows, lg, ncu);
    switch (lg.Dk) {
        case 16: launch_gdn_dk<16>(st, lraw, lrep, njobs, jobs, gp, lg, state, core, few); break;
        case 32: launch_gdn_dk<32>(st, lraw, lrep, njobs, jobs, gp, lg, state, core, few); break;
        case 64: launch_gdn_dk<64>(st, lraw, lrep, njobs, jobs, gp, lg, state, core, few); break;
        default: launch_gdn_dk<128>(st, lraw, lrep, njobs, jobs, gp, lg, state, core, few); break;
    }
    CHECK_LAUNCH();
}

// RMSNormGated (model.js:523-524: rmsnorm over each value head's Dv values
// with gated_norm, then silu_mul(z, normed)) into the out_proj operand. One
// wave per (row, value head), 8 columns a lane.
__global__ __launch_bounds__(256) void k_lin_norm(const float* __restrict__ core, const float* __restrict__ lraw,
                                                  const float* __restrict__ gnorm, float eps, int M, LinGeom lg,
                                                  int KU, uint4* __restrict__ Xp) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int h = blockIdx.x * 4 + wave, m = blockIdx.y;
    if (h >= lg.nV || m >= M) return;
    const int d0 = 8 * lane;
    const bool act = d0 < lg.Dv;
    float v[8];
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        v[j] = act ? core[(size_t)m * lg.valueDim + h * lg.Dv + d0 + j] : 0.0f;
        ss += v[j] * v[j];
    }
    ss = wave_sum(ss);
    if (!act) return;
    const float scale = 1.0f / sqrtf(ss / (float)lg.Dv + eps);
    const float* z = lraw + (size_t)m * lg.W + lg.convDim + h * lg.Dv + d0;
    float o[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const float y = v[j] * scale * gnorm[d0 + j];
        const float sg = 1.0f / (1.0f + expf(-z[j]));
        o[j] = z[j] * sg * y;
    }
    write_hilo(Xp, m, (h * lg.Dv + d0) >> 3, KU, o);
}

void launch_lin_norm(hipStream_t st, const float* core, const float* lraw, const float* gnorm, float eps, int M,
                     const LinGeom& lg, int KU, uint4* Xp) {
    if (M <= 0) return;
    hipLaunchKernelGGL(k_lin_norm, dim3((lg.nV + 3) / 4, M), dim3(256), 0, st, core, lraw, gnorm, eps, M, lg, KU, Xp);
    CHECK_LAUNCH();
}

// ================================================================ attention ===
// Ragged GQA attention over each chat's own int8 pages
// (web/model/kernels.js:1140-1310 qk_scores_gqa, causal_softmax, attn_av_gqa,
// driven per segment by web/model/model.js:321-351). Every K/V byte of a kv
// head is read once for all the job's query rows rho = i*group + gi of it:
//   S^T[token][rho] = sum_g sk[token][g] * (K_g . Qhi_g + K_g . Qlo_g) on MFMA,
//   masked to token < T_act and token <= past + i (causal inside a verify or
//   prefill run), scaled by 1/sqrt(D);
//   O^T[d][rho] += V^T[d][token] . (p * sv[token][d/32]) (hi/lo) on MFMA.
// The reference's softmax is exact three-pass; this one is online (per page)
// with a log-sum-exp merge of the chunks, equal within tolerance.
// Attention, one wave per work item: (job, kv head, query m-tile, chunk of
// `ppw` pages). The wave walks its pages in order and keeps an online softmax
// (running max, sum, rescaled O) across them; its (max, sum, O) partial for
// the 16 query rows goes to `part` (16 rows of D + 4 floats: max in log2
// units, sum, two pad floats, O). Per page: S^T = K . Q^T (hi/lo)
// scaled per (token, 32-block), masked (token < T_act, token <= past + i) and
// scaled by 1/sqrt(D); O^T += V^T . (p * sv) (hi/lo).
//
// Latency: as soon as S is formed the wave issues the next page's loads — its
// K and V scale blocks (1 KiB each, 16 B a lane into registers, written to
// the wave's LDS slice when that page starts), then its K codes into the K
// registers — and after the PV products the next page's V codes into the V
// registers. So one page of codes is held in registers (two waves per SIMD),
// and no load waits at its point of use. (Loading the scales straight into
// LDS instead makes the compiler wait for those in-flight loads before any
// LDS read it cannot prove apart from them.) Scheduling barriers keep the
// compiler from hoisting the V dequantisation into the S phase, which would
// make S wait for the V loads.
// Every page is read through a buffer resource whose base is that page's
// (page, kv head) block (64-bit address arithmetic, so pools may exceed
// 4 GB) and whose size is the block: an offset outside it reads zero.
// At head_dim <= 128 the K and V code loads are non-temporal (cache policy
// nt): a pass reads each page's codes once, and streaming them leaves the L2
// to what the kernels after attention read (measured: the whole pass
// 0.4-1.3% faster at 32 one-row chats and 0.7-0.8% at 16 verify jobs of 8
// rows, although the attention launch alone is slower). At head_dim 256 (one
// wave a SIMD) they measured 2-3% slower for the whole pass and stay
// ordinary loads, as do the 1 KiB scale blocks (non-temporal: no better).
//
// Every lane builds its fragments and rescales O on every page, with no
// branch on row state: MFMA reads all lanes' operands whatever the execution
// mask, and a still fully masked row (max -inf) just takes alpha = 0, p = 0.
// One work item of a wave: its (job, kv head, m-tile) over the chunk's pages,
// with the wave's LDS slices for the page's K and V scale blocks.
// Whether any of four V scales (f32 bits) is too large for the shifted P.V
// split (p * s * PV_SHIFT would overflow f16) — or not finite.
__device__ static inline bool pv_big(u32x4 v) {
    bool b = false;
#pragma unroll
    for (int e = 0; e < 4; e++) b = b || !(__uint_as_float(v[e]) <= PV_SCALE_MAX);
    return b;
}

template <int NG>
__device__ __forceinline__ void attn_item(const AttnItem& it, const uint4* __restrict__ Qp,
                                          const uint8_t* __restrict__ kpool, const uint8_t* __restrict__ vpool,
                                          const uint32_t* __restrict__ page_table, const KVGeom& g, int group,
                                          int ppw, float* __restrict__ part, float* ksl_w, float* vsl_w) {
    constexpr int D = 32 * NG;
    constexpr int DT = D / 16;
    constexpr int SCL = NG > 4 ? NG / 4 : 1;   // 1 KiB loads per scale block (16 B a lane)
    const int lane = threadIdx.x & 63, j4 = lane >> 4, l16 = lane & 15;
    const int T_act = it.past + it.n;
    const int R = it.n * group;
    const int npg = (T_act + 63) >> 6;
    const int p0 = it.p0;
    const int p1 = min(npg, p0 + ppw);
    const int mtq = it.mt;
    // scores in log2 units: exp(s/sqrt(D)) = exp2(s * log2(e)/sqrt(D)), one v_exp_f32 each
    const float score_scale = 1.4426950408889634f / sqrtf((float)D);

    uint4 qh[NG], ql[NG];
    {
        const size_t qb = (size_t)it.qb + lane;
#pragma unroll
        for (int gg = 0; gg < NG; gg++) {
            qh[gg] = Qp[qb + (size_t)gg * 128];
            ql[gg] = Qp[qb + (size_t)gg * 128 + 64];
        }
    }
    const int rho = mtq * 16 + l16;
    const int lim = rho < R ? it.past + rho / group : -1;   // last visible token of this row
    const uint32_t* pt = page_table + (size_t)it.slot * g.max_pages;
    const size_t hoff = (size_t)it.kvh * g.blk;
    const size_t pstride = (size_t)g.nKV * g.blk;
    // The chunk's page indices, one a lane (ppw <= 64): a page reads its own
    // with v_readlane, so no memory access sits on the page-to-page path.
    const uint32_t pgv = lane < p1 - p0 ? pt[p0 + lane] : 0u;
    auto page_rsrc = [&](const uint8_t* pool, int p) {
        const uint32_t pg = __builtin_amdgcn_readlane(pgv, p - p0);
        return __builtin_amdgcn_make_buffer_rsrc((void*)(pool + (size_t)pg * pstride + hoff), 0, g.blk, 0x00020000);
    };
    // Lane offsets inside a block (layout of k_fin_qkv's writes):
    const int vk = l16 * D + (D / 4) * j4;   // K codes: token row l16 of a 16-token tile, lane's k-block
    const int vv = j4 * D * 16 + l16 * 16;   // V codes: lane's token block, channel l16 of a d-tile
    // Scale blocks sit at 64*D in both blocks: K [64 tokens][NG], V [4][NG][16] at vpos.
    // The V scales go to LDS as [NG][4][16]: the four token blocks a wave reads
    // at once then sit in different banks. Each lane loads the 16 bytes it
    // stores at its own LDS offset, so the stores are contiguous as well.
    int vso[SCL];
#pragma unroll
    for (int q = 0; q < SCL; q++) {
        const int e = 256 * q + lane * 4, b = e >> 6, jb = (e >> 4) & 3;
        vso[q] = 4 * ((jb * NG + b) * 16 + (e & 15));
    }

    float mrow = -INFINITY, lsum = 0.0f;
    bool shifted = true;   // this row's p carries 2^PV_SHIFT_LOG2 (its O and lsum too) until dropped
    float4_t o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++) o[dt] = float4_t{0.f, 0.f, 0.f, 0.f};

    u32x4 kc[4][NG / 2], vc[DT];
    u32x4 kst[SCL], vst[SCL];   // the next page's scale blocks, 16 B a lane per KiB, on their way to LDS
    // the next page's scale blocks, then its K codes
    auto load_k = [&](__amdgpu_buffer_rsrc_t rk, __amdgpu_buffer_rsrc_t rv) {
#pragma unroll
        for (int q = 0; q < SCL; q++) {
            kst[q] = __builtin_amdgcn_raw_buffer_load_b128(rk, lane * 16, 64 * D + 1024 * q, 0);
            vst[q] = __builtin_amdgcn_raw_buffer_load_b128(rv, vso[q], 64 * D, 0);
        }
#pragma unroll
        for (int tt = 0; tt < 4; tt++)
#pragma unroll
            for (int q = 0; q < NG / 2; q++)
                kc[tt][q] = __builtin_amdgcn_raw_buffer_load_b128(rk, vk, tt * 16 * D + 16 * q, NG > 4 ? 0 : 2);
    };
    auto load_v = [&](__amdgpu_buffer_rsrc_t rv) {
#pragma unroll
        for (int dt = 0; dt < DT; dt++) vc[dt] = __builtin_amdgcn_raw_buffer_load_b128(rv, vv, dt * 256, NG > 4 ? 0 : 2);
    };
    // One page. Its scale blocks arrived in kst/vst during the previous page;
    // they go to this wave's LDS slice first (a wave's LDS accesses run in
    // order, so the previous page's reads of the slice are done). The V
    // scales of tokens past the job's are another session's stale values
    // (even NaN): they go in as zero, so p * s is zero for every token whose
    // p is (a masked token's p is exp2(-inf) = +0, every scale of a visible
    // token is finite and positive).
    auto page = [&](int p) {
        // the last page reloads itself instead of branching (an L2 hit)
        const int pn = p + 1 < p1 ? p + 1 : p;
        bool big = false;
#pragma unroll
        for (int q = 0; q < SCL; q++) {
            *(u32x4*)&ksl_w[256 * q + lane * 4] = kst[q];
            u32x4 v = vst[q];
            if (p * 64 + 64 > T_act) {
                // LDS element 256q + 4 lane + e holds V position v = 16 jj + 4 (lane & 3) + e,
                // jj = ((256q + 4 lane) >> 4) & 3: the page's token vpos(v) = 16 (lane & 3) + 4 jj + e
                const int t0 = p * 64 + 16 * (lane & 3) + 4 * (((256 * q + lane * 4) >> 4) & 3);
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (t0 + e >= T_act) v[e] = 0u;
            }
            big = big || pv_big(v);
            *(u32x4*)&vsl_w[256 * q + lane * 4] = v;
        }
        const bool pbig = __builtin_amdgcn_ballot_w64(big) != 0;
        {
            float pr[4][4];
            float pm = -INFINITY;
#pragma unroll
            for (int tt = 0; tt < 4; tt++) {
                float ks[4 * NG];   // tokens 16tt + 4j4 + r, groups 0..NG-1
#pragma unroll
                for (int q = 0; q < NG; q++) {
                    const float4 f = *(const float4*)&ksl_w[(tt * 16 + 4 * j4) * NG + 4 * q];
                    ks[4 * q] = f.x; ks[4 * q + 1] = f.y; ks[4 * q + 2] = f.z; ks[4 * q + 3] = f.w;
                }
                float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int gg = 0; gg < NG; gg++) {
                    const u32x4 c = kc[tt][gg >> 1];
                    const half8_t kf = (gg & 1) ? dequant8_biased(c[2], c[3]) : dequant8_biased(c[0], c[1]);
                    float4_t pp = {0.f, 0.f, 0.f, 0.f};
                    pp = mfma16x16x32(kf, __builtin_bit_cast(half8_t, qh[gg]), pp);
                    pp = mfma16x16x32(kf, __builtin_bit_cast(half8_t, ql[gg]), pp);
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[r] = __builtin_fmaf(ks[r * NG + gg], pp[r], acc[r]);
                }
#pragma unroll
                for (int r = 0; r < 4; r++) pr[tt][r] = acc[r] * score_scale;
            }
            // every token up to the job's first new position is visible to every
            // query row (and below T_act): only a page past it needs the per-cell
            // mask. The m-tile's lanes past the job's rows then carry unmasked
            // scores; they stay in their own lanes and MFMA columns, never written.
            if (p * 64 + 63 > it.past) {
#pragma unroll
                for (int tt = 0; tt < 4; tt++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int tok = p * 64 + tt * 16 + 4 * j4 + r;
                        if (!(tok < T_act && tok <= lim)) pr[tt][r] = -INFINITY;
                    }
            }
#pragma unroll
            for (int tt = 0; tt < 4; tt++)
#pragma unroll
                for (int r = 0; r < 4; r++) pm = fmaxf(pm, pr[tt][r]);
            const auto rvn = page_rsrc(vpool, pn);
            load_k(page_rsrc(kpool, pn), rvn);   // the K registers are free: start the next page
            __builtin_amdgcn_sched_barrier(0);
            pm = fmaxf(pm, __shfl_xor(pm, 16));
            pm = fmaxf(pm, __shfl_xor(pm, 32));
            const float mnew = fmaxf(mrow, pm);
            // the row drops the shift for good on a page whose V scales or its own
            // running max (in log2 units) leave no f16 room for p * s
            const bool drop = pbig || !(fabsf(mnew) < PV_MAX_SCORE);
            const float shrink = drop && shifted ? PV_UNSHIFT : 1.0f;
            shifted = shifted && !drop;
            const float alpha = (mrow == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mrow - mnew)) * shrink;
            lsum *= alpha;
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int r = 0; r < 4; r++) o[dt][r] *= alpha;
            const float msub = (mnew == -INFINITY ? 0.0f : mnew) - (shifted ? PV_SHIFT_LOG2 : 0.0f);
#pragma unroll
            for (int tt = 0; tt < 4; tt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float e = __builtin_amdgcn_exp2f(pr[tt][r] - msub);   // masked: exp2(-inf) = 0
                    pr[tt][r] = e;
                    lsum += e;
                }
            __builtin_amdgcn_sched_barrier(0);
            // p * s (p times 2^PV_SHIFT_LOG2 while shifted) as hi + lo (split_hilo2), both into O
#pragma unroll
            for (int b = 0; b < NG; b++) {
                float sv[16];   // the lane's 16 tokens of 32-block b
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float4 f = *(const float4*)&vsl_w[b * 64 + 16 * j4 + 4 * q];
                    sv[4 * q] = f.x; sv[4 * q + 1] = f.y; sv[4 * q + 2] = f.z; sv[4 * q + 3] = f.w;
                }
#pragma unroll
                for (int ks = 0; ks < 2; ks++) {
                    u32x4 phw, plw;
#pragma unroll
                    for (int ii = 0; ii < 8; ii += 2) {
                        const int tt = 2 * ks + (ii >> 2), r = ii & 3;
                        const float p0 = pr[tt][r] * sv[4 * tt + r];
                        const float p1 = pr[tt][r + 1] * sv[4 * tt + r + 1];
                        uint32_t h, l;
                        split_hilo2(p0, p1, h, l);
                        phw[ii >> 1] = h;
                        plw[ii >> 1] = l;
                    }
                    const half8_t ph = __builtin_bit_cast(half8_t, phw), pl = __builtin_bit_cast(half8_t, plw);
#pragma unroll
                    for (int dd = 0; dd < 2; dd++) {
                        const int dt = 2 * b + dd;
                        const u32x4 c = vc[dt];
                        const half8_t vf = ks ? dequant8_biased(c[2], c[3]) : dequant8_biased(c[0], c[1]);
                        o[dt] = mfma16x16x32(vf, ph, o[dt]);
                        o[dt] = mfma16x16x32(vf, pl, o[dt]);
                    }
                }
            }
            mrow = mnew;
            load_v(rvn);
        }
    };
    if (p0 < p1) {
        const auto rv = page_rsrc(vpool, p0);
        load_k(page_rsrc(kpool, p0), rv);
        load_v(rv);
        for (int p = p0; p < p1; p++) page(p);
    }
    lsum += __shfl_xor(lsum, 16);
    lsum += __shfl_xor(lsum, 32);
    // partial row: max, sum, two pad floats, then O (16-byte aligned), the
    // shift taken off; rows past the job's R query rows are neither written
    // nor read
    if (rho < R) {
        const float un = shifted ? PV_UNSHIFT : 1.0f;
        float* dst = part + it.part + (size_t)l16 * (D + 4);
#pragma unroll
        for (int dt = 0; dt < DT; dt++) *(float4_t*)(dst + 4 + dt * 16 + 4 * j4) = o[dt] * un;
        if (j4 == 0) *(float2*)dst = make_float2(mrow, lsum * un);
    }
}


// One block of a job of several m-tiles: its four waves hold m-tiles
// 4b .. 4b+3 of one (job, kv head, chunk) (an m-tile past the job's is an
// empty slot, mt < 0) and read the same pages. Each wave loads a quarter of
// a page (K token tile w, V d-tiles w*DT/4 ..), dequantises it once into the
// workgroup's LDS, and every wave's MFMAs read the fragments from there, so a
// page is dequantised once instead of once per m-tile; a block with an empty
// slot has its idle wave 3 load and dequantise the whole page instead, while
// the other waves only compute. One barrier a page;
// the fragments are double-buffered (a wave past page p's barrier has
// finished page p - 1, so page p + 1 may reuse that buffer). Every value and
// every operation of a row is the one attn_item computes for it.
template <int NG>
__device__ __forceinline__ void attn_block4(const AttnItem& it, const AttnItem& it0, int wv,
                                            const uint4* __restrict__ Qp, const uint8_t* __restrict__ kpool,
                                            const uint8_t* __restrict__ vpool,
                                            const uint32_t* __restrict__ page_table, const KVGeom& g, int group,
                                            int ppw, float* __restrict__ part, u32x4* lds) {
    constexpr int D = 32 * NG;
    constexpr int DT = D / 16, DQ = DT / 4;
    constexpr int SCL = NG > 4 ? NG / 4 : 1;
    // LDS: K fragments [2][4 tt][NG gg][64], V fragments [2][DT][2 ks][64], then the
    // K and V scale blocks [2][256 * SCL] floats each, then the pages' range flags [2]
    u32x4* kf_s = lds;
    u32x4* vf_s = kf_s + 2 * 4 * NG * 64;
    float* ks_s = (float*)(vf_s + 2 * DT * 2 * 64);
    float* vs_s = ks_s + 2 * 256 * SCL;
    int* big_s = (int*)(vs_s + 2 * 256 * SCL);   // [2]: the page's V scales forbid the P.V shift
    const int lane = threadIdx.x & 63, j4 = lane >> 4, l16 = lane & 15;
    const int T_act = it0.past + it0.n;
    const int R = it0.n * group;
    const int npg = (T_act + 63) >> 6;
    const int p0 = it0.p0;
    const int p1 = min(npg, p0 + ppw);
    const bool mine = it.mt >= 0;
    const float score_scale = 1.4426950408889634f / sqrtf((float)D);

    uint4 qh[NG], ql[NG];
    if (mine) {
        const size_t qb = (size_t)it.qb + lane;
#pragma unroll
        for (int gg = 0; gg < NG; gg++) {
            qh[gg] = Qp[qb + (size_t)gg * 128];
            ql[gg] = Qp[qb + (size_t)gg * 128 + 64];
        }
    }
    const int rho = (mine ? it.mt : 0) * 16 + l16;
    const int lim = mine && rho < R ? it0.past + rho / group : -1;
    const uint32_t* pt = page_table + (size_t)it0.slot * g.max_pages;
    const size_t hoff = (size_t)it0.kvh * g.blk;
    const size_t pstride = (size_t)g.nKV * g.blk;
    const uint32_t pgv = lane < p1 - p0 ? pt[p0 + lane] : 0u;
    auto page_rsrc = [&](const uint8_t* pool, int p) {
        const uint32_t pg = __builtin_amdgcn_readlane(pgv, p - p0);
        return __builtin_amdgcn_make_buffer_rsrc((void*)(pool + (size_t)pg * pstride + hoff), 0, g.blk, 0x00020000);
    };
    const int vk = l16 * D + (D / 4) * j4;
    const int vv = j4 * D * 16 + l16 * 16;
    int vso[SCL];
#pragma unroll
    for (int q = 0; q < SCL; q++) {
        const int e = 256 * q + lane * 4, b = e >> 6, jb = (e >> 4) & 3;
        vso[q] = 4 * ((jb * NG + b) * 16 + (e & 15));
    }

    float mrow = -INFINITY, lsum = 0.0f;
    bool shifted = true;   // as in attn_item
    float4_t o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++) o[dt] = float4_t{0.f, 0.f, 0.f, 0.f};

    // this wave's quarter of the next page: K token tile wv, V d-tiles wv*DQ .. +DQ-1,
    // and (waves 0 and 1) the K or V scale block
    u32x4 kc[NG / 2], vc[DQ], sc[SCL];
    auto load = [&](int p) {
        const auto rk = page_rsrc(kpool, p), rv = page_rsrc(vpool, p);
#pragma unroll
        for (int q = 0; q < NG / 2; q++) kc[q] = __builtin_amdgcn_raw_buffer_load_b128(rk, vk, wv * 16 * D + 16 * q, NG > 4 ? 0 : 2);
#pragma unroll
        for (int i = 0; i < DQ; i++) vc[i] = __builtin_amdgcn_raw_buffer_load_b128(rv, vv, (wv * DQ + i) * 256, NG > 4 ? 0 : 2);
        if (wv == 0) {
#pragma unroll
            for (int q = 0; q < SCL; q++) sc[q] = __builtin_amdgcn_raw_buffer_load_b128(rk, lane * 16, 64 * D + 1024 * q, 0);
        } else if (wv == 1) {
#pragma unroll
            for (int q = 0; q < SCL; q++) sc[q] = __builtin_amdgcn_raw_buffer_load_b128(rv, vso[q], 64 * D, 0);
        }
    };
    // A block with an empty slot (a job of 3 m-tiles or fewer in its last
    // block, as a verify of 8 rows x 5 heads) gives its idle wave 3 the whole
    // page: it loads and dequantises everything, the same fragments the four
    // quarters would be, while the other waves only compute. Its page loop
    // has the same barriers as theirs.
    const int mtq = (it0.n * group + 15) >> 4;
    const bool spare = mtq - it0.mt < 4;
    if (spare && wv == 3) {
        u32x4 fk[4][NG / 2], fv[DT], fs[2][SCL];
        auto load_all = [&](int p) {
            const auto rk = page_rsrc(kpool, p), rv = page_rsrc(vpool, p);
#pragma unroll
            for (int tt = 0; tt < 4; tt++)
#pragma unroll
                for (int q = 0; q < NG / 2; q++)
                    fk[tt][q] = __builtin_amdgcn_raw_buffer_load_b128(rk, vk, tt * 16 * D + 16 * q, NG > 4 ? 0 : 2);
#pragma unroll
            for (int dt = 0; dt < DT; dt++) fv[dt] = __builtin_amdgcn_raw_buffer_load_b128(rv, vv, dt * 256, NG > 4 ? 0 : 2);
#pragma unroll
            for (int q = 0; q < SCL; q++) {
                fs[0][q] = __builtin_amdgcn_raw_buffer_load_b128(rk, lane * 16, 64 * D + 1024 * q, 0);
                fs[1][q] = __builtin_amdgcn_raw_buffer_load_b128(rv, vso[q], 64 * D, 0);
            }
        };
        if (p0 < p1) load_all(p0);
        for (int p = p0; p < p1; p++) {
            const int B = (p - p0) & 1;
            u32x4* kf = kf_s + B * 4 * NG * 64;
            u32x4* vf = vf_s + B * DT * 2 * 64;
            float* ksl = ks_s + B * 256 * SCL;
            float* vsl = vs_s + B * 256 * SCL;
#pragma unroll
            for (int tt = 0; tt < 4; tt++)
#pragma unroll
                for (int q = 0; q < NG / 2; q++) {
                    kf[(tt * NG + 2 * q) * 64 + lane] = __builtin_bit_cast(u32x4, dequant8_biased(fk[tt][q][0], fk[tt][q][1]));
                    kf[(tt * NG + 2 * q + 1) * 64 + lane] =
                        __builtin_bit_cast(u32x4, dequant8_biased(fk[tt][q][2], fk[tt][q][3]));
                }
#pragma unroll
            for (int dt = 0; dt < DT; dt++) {
                vf[(dt * 2) * 64 + lane] = __builtin_bit_cast(u32x4, dequant8_biased(fv[dt][0], fv[dt][1]));
                vf[(dt * 2 + 1) * 64 + lane] = __builtin_bit_cast(u32x4, dequant8_biased(fv[dt][2], fv[dt][3]));
            }
            bool big = false;
#pragma unroll
            for (int q = 0; q < SCL; q++) {
                *(u32x4*)&ksl[256 * q + lane * 4] = fs[0][q];
                u32x4 v = fs[1][q];
                if (p * 64 + 64 > T_act) {
                    const int t0 = p * 64 + 16 * (lane & 3) + 4 * (((256 * q + lane * 4) >> 4) & 3);
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (t0 + e >= T_act) v[e] = 0u;
                }
                big = big || pv_big(v);
                *(u32x4*)&vsl[256 * q + lane * 4] = v;
            }
            const bool pbig = __builtin_amdgcn_ballot_w64(big) != 0;
            if (lane == 0) big_s[B] = pbig ? 1 : 0;
            __syncthreads();
            if (p + 1 < p1) load_all(p + 1);
        }
        return;   // wave 3's slot is empty
    }
    if (p0 < p1 && !spare) load(p0);
    for (int p = p0; p < p1; p++) {
        const int B = (p - p0) & 1;
        u32x4* kf = kf_s + B * 4 * NG * 64;
        u32x4* vf = vf_s + B * DT * 2 * 64;
        float* ksl = ks_s + B * 256 * SCL;
        float* vsl = vs_s + B * 256 * SCL;
        if (!spare) {
#pragma unroll
            for (int q = 0; q < NG / 2; q++) {
                kf[(wv * NG + 2 * q) * 64 + lane] = __builtin_bit_cast(u32x4, dequant8_biased(kc[q][0], kc[q][1]));
                kf[(wv * NG + 2 * q + 1) * 64 + lane] = __builtin_bit_cast(u32x4, dequant8_biased(kc[q][2], kc[q][3]));
            }
#pragma unroll
            for (int i = 0; i < DQ; i++) {
                vf[((wv * DQ + i) * 2) * 64 + lane] = __builtin_bit_cast(u32x4, dequant8_biased(vc[i][0], vc[i][1]));
                vf[((wv * DQ + i) * 2 + 1) * 64 + lane] = __builtin_bit_cast(u32x4, dequant8_biased(vc[i][2], vc[i][3]));
            }
            if (wv == 0) {
#pragma unroll
                for (int q = 0; q < SCL; q++) *(u32x4*)&ksl[256 * q + lane * 4] = sc[q];
            } else if (wv == 1) {
                bool big = false;
#pragma unroll
                for (int q = 0; q < SCL; q++) {
                    u32x4 v = sc[q];
                    if (p * 64 + 64 > T_act) {   // stale scales past the job's tokens go in as zero
                        const int t0 = p * 64 + 16 * (lane & 3) + 4 * (((256 * q + lane * 4) >> 4) & 3);
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            if (t0 + e >= T_act) v[e] = 0u;
                    }
                    big = big || pv_big(v);
                    *(u32x4*)&vsl[256 * q + lane * 4] = v;
                }
                const bool pbig = __builtin_amdgcn_ballot_w64(big) != 0;
                if (lane == 0) big_s[B] = pbig ? 1 : 0;
            }
        }
        __syncthreads();
        if (p + 1 < p1 && !spare) load(p + 1);   // the registers are free: the next page is on its way
        if (!mine) continue;
        float pr[4][4];
        float pm = -INFINITY;
#pragma unroll
        for (int tt = 0; tt < 4; tt++) {
            float ks[4 * NG];
#pragma unroll
            for (int q = 0; q < NG; q++) {
                const float4 f = *(const float4*)&ksl[(tt * 16 + 4 * j4) * NG + 4 * q];
                ks[4 * q] = f.x; ks[4 * q + 1] = f.y; ks[4 * q + 2] = f.z; ks[4 * q + 3] = f.w;
            }
            float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int gg = 0; gg < NG; gg++) {
                const half8_t kfr = __builtin_bit_cast(half8_t, kf[(tt * NG + gg) * 64 + lane]);
                float4_t pp = {0.f, 0.f, 0.f, 0.f};
                pp = mfma16x16x32(kfr, __builtin_bit_cast(half8_t, qh[gg]), pp);
                pp = mfma16x16x32(kfr, __builtin_bit_cast(half8_t, ql[gg]), pp);
#pragma unroll
                for (int r = 0; r < 4; r++) acc[r] = __builtin_fmaf(ks[r * NG + gg], pp[r], acc[r]);
            }
#pragma unroll
            for (int r = 0; r < 4; r++) pr[tt][r] = acc[r] * score_scale;
        }
        // every token up to the job's first new position is visible to every
        // query row (and below T_act): only a page past it needs the per-cell
        // mask. The m-tile's lanes past the job's rows then carry unmasked
        // scores; they stay in their own lanes and MFMA columns, never written.
        if (p * 64 + 63 > it0.past) {
#pragma unroll
            for (int tt = 0; tt < 4; tt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int tok = p * 64 + tt * 16 + 4 * j4 + r;
                    if (!(tok < T_act && tok <= lim)) pr[tt][r] = -INFINITY;
                }
        }
#pragma unroll
        for (int tt = 0; tt < 4; tt++)
#pragma unroll
            for (int r = 0; r < 4; r++) pm = fmaxf(pm, pr[tt][r]);
        pm = fmaxf(pm, __shfl_xor(pm, 16));
        pm = fmaxf(pm, __shfl_xor(pm, 32));
        const float mnew = fmaxf(mrow, pm);
        const bool pbig = __builtin_amdgcn_readfirstlane(big_s[B]) != 0;
        const bool drop = pbig || !(fabsf(mnew) < PV_MAX_SCORE);   // as in attn_item
        const float shrink = drop && shifted ? PV_UNSHIFT : 1.0f;
        shifted = shifted && !drop;
        const float alpha = (mrow == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mrow - mnew)) * shrink;
        lsum *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int r = 0; r < 4; r++) o[dt][r] *= alpha;
        const float msub = (mnew == -INFINITY ? 0.0f : mnew) - (shifted ? PV_SHIFT_LOG2 : 0.0f);
#pragma unroll
        for (int tt = 0; tt < 4; tt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float e = __builtin_amdgcn_exp2f(pr[tt][r] - msub);
                pr[tt][r] = e;
                lsum += e;
            }
#pragma unroll
        for (int b = 0; b < NG; b++) {
            float sv[16];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float4 f = *(const float4*)&vsl[b * 64 + 16 * j4 + 4 * q];
                sv[4 * q] = f.x; sv[4 * q + 1] = f.y; sv[4 * q + 2] = f.z; sv[4 * q + 3] = f.w;
            }
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                u32x4 phw, plw;
#pragma unroll
                for (int ii = 0; ii < 8; ii += 2) {
                    const int tt = 2 * ks + (ii >> 2), r = ii & 3;
                    uint32_t h, l;
                    split_hilo2(pr[tt][r] * sv[4 * tt + r], pr[tt][r + 1] * sv[4 * tt + r + 1], h, l);
                    phw[ii >> 1] = h;
                    plw[ii >> 1] = l;
                }
                const half8_t ph = __builtin_bit_cast(half8_t, phw), pl = __builtin_bit_cast(half8_t, plw);
#pragma unroll
                for (int dd = 0; dd < 2; dd++) {
                    const int dt = 2 * b + dd;
                    const half8_t vfr = __builtin_bit_cast(half8_t, vf[(dt * 2 + ks) * 64 + lane]);
                    o[dt] = mfma16x16x32(vfr, ph, o[dt]);
                    o[dt] = mfma16x16x32(vfr, pl, o[dt]);
                }
            }
        }
        mrow = mnew;
    }
    if (!mine) return;
    lsum += __shfl_xor(lsum, 16);
    lsum += __shfl_xor(lsum, 32);
    if (rho < R) {
        const float un = shifted ? PV_UNSHIFT : 1.0f;
        float* dst = part + it.part + (size_t)l16 * (D + 4);
#pragma unroll
        for (int dt = 0; dt < DT; dt++) *(float4_t*)(dst + 4 + dt * 16 + 4 * j4) = o[dt] * un;
        if (j4 == 0) *(float2*)dst = make_float2(mrow, lsum * un);
    }
}

// LDS of a k_attn workgroup: the four waves' scale slices for one-m-tile
// items (8 KiB per 4 groups), or a block's shared fragments and scales
// (attn_block4) when the launch holds jobs of several m-tiles (`multi`).
template <int NG>
constexpr size_t attn_lds_bytes() {
    constexpr size_t SCL = NG > 4 ? NG / 4 : 1, DT = 2 * NG;
    constexpr size_t single = 8 * 256 * SCL * 4;
    constexpr size_t block = (2 * 4 * NG * 64 + 2 * DT * 2 * 64) * 16 + 2 * 2 * 256 * SCL * 4 + 16;
    return single > block ? single : block;
}

// Work items go to waves in workgroups of four (item 4b + w to wave w of
// block b). Workgroup i takes block i; with `dyn` set, it then takes blocks
// gridDim.x, gridDim.x + 1, ... from the counter ctr[par] as it finishes
// each (launch_attn sets it for launches a little over one round of
// resident workgroups: dispatch hands a pending workgroup to a fixed XCD, so
// the few blocks past the first round would wait for that XCD's slowest
// workgroups). Each launch clears the counter of the next launch on its
// stream, ctr[par ^ 1]; the one it counts with was cleared by the
// launch before it. A block of one chunk's m-tiles (a job of several
// m-tiles, in a launch with `multi` set) runs attn_block4, its four waves
// sharing each page's dequantised fragments; other blocks' waves run their
// items on their own (attn_item).
template <int NG>
__global__ __launch_bounds__(256, NG > 4 ? 1 : 2) void k_attn(const AttnItem* __restrict__ items, int nitems,
                                                 const uint4* __restrict__ Qp,
                                                 const uint8_t* __restrict__ kpool, const uint8_t* __restrict__ vpool,
                                                 const uint32_t* __restrict__ page_table, KVGeom g, int group, int ppw,
                                                 float* __restrict__ part, uint32_t* __restrict__ ctr, int par,
                                                 int dyn, int multi) {
    // per wave, the current page's K and V scale blocks (64 tokens x NG groups,
    // f32), or a block's shared fragments: attn_lds_bytes<NG>() of dynamic LDS
    constexpr int SCL = NG > 4 ? NG / 4 : 1;
    extern __shared__ __attribute__((aligned(1024))) u32x4 lds[];
    __shared__ int s_blk;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (blockIdx.x == 0 && threadIdx.x == 0)
        __hip_atomic_store(&ctr[par ^ 1], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int nblk = (nitems + 3) / 4;
    for (int blk = blockIdx.x;;) {
        const int wid = blk * 4 + wv;
        const AttnItem it0 = items[blk * 4];
        if (multi && it0.n * group > 16) {
            // a job of several m-tiles: the block is one chunk's m-tiles (mt < 0 pads it)
            attn_block4<NG>(items[wid], it0, wv, Qp, kpool, vpool, page_table, g, group, ppw, part, lds);
        } else if (wid < nitems) {
            const AttnItem it = items[wid];
            if (it.mt >= 0)
                attn_item<NG>(it, Qp, kpool, vpool, page_table, g, group, ppw, part, (float*)lds + wv * 256 * SCL,
                              (float*)lds + (4 + wv) * 256 * SCL);
        }
        if (!dyn) break;   // no barriers then: a finished wave may leave
        __syncthreads();
        if (threadIdx.x == 0) s_blk = (int)gridDim.x + (int)atomicAdd(&ctr[par], 1u);
        __syncthreads();
        blk = s_blk;
        if (blk >= nblk) break;
    }
}

// Few items, each of one m-tile: a workgroup an item. Alone, a wave of
// attn_item dequantises a page's 64 x D codes twice over (K and V) in about
// 2.6 us, and a chat's chunks leave most of the GPU's SIMDs without one. Here
// wave w takes the page's K token tile w and the V d-tiles w*DT/4 .., with
// their scales straight into registers; the scores cross in LDS, one barrier
// a page (two buffers: a wave past page p's barrier has read page p - 1's),
// and every wave goes through the whole softmax. A page's share is a quarter
// of the registers, so two pages are on their way. Bound by that chain: 9000
// tokens of one chat (144 items of 8 pages, head_dim 128) 22.5 -> 14.5 us a
// launch. Every value and every operation of a row is the one attn_item
// computes for it.
template <int NG>
__global__ __launch_bounds__(256, 1) void k_attn_wide(const AttnItem* __restrict__ items, const uint4* __restrict__ Qp,
                                                      const uint8_t* __restrict__ kpool,
                                                      const uint8_t* __restrict__ vpool,
                                                      const uint32_t* __restrict__ page_table, KVGeom g, int group,
                                                      int ppw, float* __restrict__ part) {
    constexpr int D = 32 * NG, DT = D / 16, DW = DT / 4, NB = NG > 4 ? NG / 4 : 1;   // d-tiles, 32-blocks a wave
    __shared__ float4_t s_p[2][4][64];
    __shared__ int s_big[2][4];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, j4 = lane >> 4, l16 = lane & 15;
    const AttnItem it = items[blockIdx.x];
    if (it.mt < 0) return;   // the whole workgroup
    const int T_act = it.past + it.n;
    const int R = it.n * group;
    const int npg = (T_act + 63) >> 6;
    const int p0 = it.p0, p1 = min(npg, p0 + ppw);
    const float score_scale = 1.4426950408889634f / sqrtf((float)D);
    const int b0 = wv * DW / 2;   // the wave's first 32-block of V
    const uint32_t* pt = page_table + (size_t)it.slot * g.max_pages;
    const uint32_t pgv = lane < p1 - p0 ? pt[p0 + lane] : 0u;
    const size_t hoff = (size_t)it.kvh * g.blk, pstride = (size_t)g.nKV * g.blk;
    // a page past the chunk's last: a resource of no bytes, whose loads read zero
    auto page_rsrc = [&](const uint8_t* pool, int p) {
        const uint32_t pg = __builtin_amdgcn_readlane(pgv, p < p1 ? p - p0 : 0);
        return __builtin_amdgcn_make_buffer_rsrc((void*)(pool + (size_t)pg * pstride + hoff), 0, p < p1 ? g.blk : 0,
                                                 0x00020000);
    };
    const int vk = l16 * D + (D / 4) * j4, vv = j4 * D * 16 + l16 * 16;
    struct Page {
        u32x4 kc[NG / 2], ks[NG], vc[DW], vs[NB][4];
    };
    auto load_k = [&](Page& g1, int p) {
        const auto rk = page_rsrc(kpool, p);
#pragma unroll
        for (int q = 0; q < NG / 2; q++)
            g1.kc[q] = __builtin_amdgcn_raw_buffer_load_b128(rk, vk, wv * 16 * D + 16 * q, NG > 4 ? 0 : 2);
        // tokens 16 wv + 4 j4 + r, groups 0..NG-1
#pragma unroll
        for (int q = 0; q < NG; q++)
            g1.ks[q] = __builtin_amdgcn_raw_buffer_load_b128(rk, j4 * 16 * NG + 16 * q, 64 * D + wv * 64 * NG, 0);
    };
    auto load_v = [&](Page& g1, int p) {
        const auto rv = page_rsrc(vpool, p);
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                g1.vs[b][q] = __builtin_amdgcn_raw_buffer_load_b128(rv, j4 * 64 * NG + 16 * q, 64 * D + (b0 + b) * 64, 0);
#pragma unroll
        for (int i = 0; i < DW; i++)
            g1.vc[i] = __builtin_amdgcn_raw_buffer_load_b128(rv, vv, (wv * DW + i) * 256, NG > 4 ? 0 : 2);
    };
    Page pa, pb;
    load_k(pa, p0);
    load_v(pa, p0);
    load_k(pb, p0 + 1);
    load_v(pb, p0 + 1);
    uint4 qh[NG], ql[NG];
#pragma unroll
    for (int gg = 0; gg < NG; gg++) {
        qh[gg] = Qp[(size_t)it.qb + lane + (size_t)gg * 128];
        ql[gg] = Qp[(size_t)it.qb + lane + (size_t)gg * 128 + 64];
    }
    const int rho = it.mt * 16 + l16;
    const int lim = rho < R ? it.past + rho / group : -1;
    float mrow = -INFINITY, lsum = 0.0f;
    bool shifted = true;
    float4_t o[DW];
#pragma unroll
    for (int i = 0; i < DW; i++) o[i] = float4_t{0.f, 0.f, 0.f, 0.f};

    auto page = [&](Page& g1, int p, int buf) {
        // the scores of this wave's token tile
        float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int gg = 0; gg < NG; gg++) {
            const u32x4 c = g1.kc[gg >> 1];
            const half8_t kf = (gg & 1) ? dequant8_biased(c[2], c[3]) : dequant8_biased(c[0], c[1]);
            float4_t pp = {0.f, 0.f, 0.f, 0.f};
            pp = mfma16x16x32(kf, __builtin_bit_cast(half8_t, qh[gg]), pp);
            pp = mfma16x16x32(kf, __builtin_bit_cast(half8_t, ql[gg]), pp);
#pragma unroll
            for (int r = 0; r < 4; r++)
                acc[r] = __builtin_fmaf(__uint_as_float(g1.ks[(r * NG + gg) >> 2][(r * NG + gg) & 3]), pp[r], acc[r]);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) acc[r] = acc[r] * score_scale;
        if (p * 64 + 63 > it.past) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int tok = p * 64 + wv * 16 + 4 * j4 + r;
                if (!(tok < T_act && tok <= lim)) acc[r] = -INFINITY;
            }
        }
        s_p[buf][wv][lane] = acc;
        load_k(g1, p + 2);
        bool big = false;
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                if (p * 64 + 64 > T_act) {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (p * 64 + 16 * q + 4 * j4 + e >= T_act) g1.vs[b][q][e] = 0u;
                }
                big = big || pv_big(g1.vs[b][q]);
            }
        const bool wbig = __builtin_amdgcn_ballot_w64(big) != 0;
        if (lane == 0) s_big[buf][wv] = wbig;
        __syncthreads();
        float pr[4][4];
        float pm = -INFINITY;
        bool pbig = false;
#pragma unroll
        for (int tt = 0; tt < 4; tt++) {
            const float4_t v = s_p[buf][tt][lane];
            pbig = pbig || s_big[buf][tt] != 0;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                pr[tt][r] = v[r];
                pm = fmaxf(pm, pr[tt][r]);
            }
        }
        pm = fmaxf(pm, __shfl_xor(pm, 16));
        pm = fmaxf(pm, __shfl_xor(pm, 32));
        const float mnew = fmaxf(mrow, pm);
        const bool drop = pbig || !(fabsf(mnew) < PV_MAX_SCORE);
        const float shrink = drop && shifted ? PV_UNSHIFT : 1.0f;
        shifted = shifted && !drop;
        const float alpha = (mrow == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mrow - mnew)) * shrink;
        lsum *= alpha;
#pragma unroll
        for (int i = 0; i < DW; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) o[i][r] *= alpha;
        const float msub = (mnew == -INFINITY ? 0.0f : mnew) - (shifted ? PV_SHIFT_LOG2 : 0.0f);
#pragma unroll
        for (int tt = 0; tt < 4; tt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float e = __builtin_amdgcn_exp2f(pr[tt][r] - msub);
                pr[tt][r] = e;
                lsum += e;
            }
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                u32x4 phw, plw;
#pragma unroll
                for (int ii = 0; ii < 8; ii += 2) {
                    const int tt = 2 * ks + (ii >> 2), r = ii & 3;
                    uint32_t h, l;
                    split_hilo2(pr[tt][r] * __uint_as_float(g1.vs[b][tt][r]),
                                pr[tt][r + 1] * __uint_as_float(g1.vs[b][tt][r + 1]), h, l);
                    phw[ii >> 1] = h;
                    plw[ii >> 1] = l;
                }
                const half8_t ph = __builtin_bit_cast(half8_t, phw), pl = __builtin_bit_cast(half8_t, plw);
#pragma unroll
                for (int i = b * DW / NB; i < (b + 1) * DW / NB; i++) {
                    const u32x4 c = g1.vc[i];
                    const half8_t vf = ks ? dequant8_biased(c[2], c[3]) : dequant8_biased(c[0], c[1]);
                    o[i] = mfma16x16x32(vf, ph, o[i]);
                    o[i] = mfma16x16x32(vf, pl, o[i]);
                }
            }
        mrow = mnew;
        load_v(g1, p + 2);
    };
    for (int p = p0; p < p1; p += 2) {
        page(pa, p, 0);
        if (p + 1 < p1) page(pb, p + 1, 1);
    }
    lsum += __shfl_xor(lsum, 16);
    lsum += __shfl_xor(lsum, 32);
    if (rho < R) {
        const float un = shifted ? PV_UNSHIFT : 1.0f;
        float* dst = part + it.part + (size_t)l16 * (D + 4);
#pragma unroll
        for (int i = 0; i < DW; i++) *(float4_t*)(dst + 4 + (wv * DW + i) * 16 + 4 * j4) = o[i] * un;
        if (wv == 0 && j4 == 0) *(float2*)dst = make_float2(mrow, lsum * un);
    }
}

void launch_attn(hipStream_t st, const AttnItem* items, int nitems, const uint4* Qp,
                 const uint8_t* kpool, const uint8_t* vpool, const uint32_t* page_table, const KVGeom& g, int group,
                 int ppw, float* part, int multi, AttnSched& sc) {
    if (nitems <= 0) return;
    // A workgroup an item while all are resident at once with a SIMD to each
    // wave (head_dim 256, 64) or with two waves a SIMD (128). An attention
    // launch here against k_attn's, us: head_dim 256, 32-256 items -10 to -18,
    // 288 +10; head_dim 128, 32-256 items -7 to -8, 288-512 -4 to -2, 576 +6;
    // head_dim 64 (items of 2 pages) 36-240 items -0.4 to -1.7, 258-516 within
    // 0.6 either way, 576 +2.
    if (!multi && nitems <= (g.ng == 4 ? 2 : 1) * sc.ncu) {
        const auto kern = g.ng == 8 ? k_attn_wide<8> : g.ng == 4 ? k_attn_wide<4> : k_attn_wide<2>;
        hipLaunchKernelGGL(kern, dim3(nitems), dim3(256), 0, st, items, Qp, kpool, vpool, page_table, g, group, ppw,
                           part);
        CHECK_LAUNCH();
        return;
    }
    const int nblk = (nitems + 3) / 4;
    const int cap = sc.ncu * (g.ng == 8 ? 1 : 2);   // workgroups resident at once
    // blocks past the first round go out from the counter while they are few;
    // with more, dispatch's own rounds balance them
    const int dyn = nblk > cap && 2 * nblk <= 3 * cap;
    const int blocks = dyn ? cap : nblk;
    const int par = (int)(sc.seq++ & 1u);
    static bool attr = false;
    if (!attr) {
        attr = true;
        (void)hipFuncSetAttribute((const void*)k_attn<8>, hipFuncAttributeMaxDynamicSharedMemorySize, attn_lds_bytes<8>());
        (void)hipFuncSetAttribute((const void*)k_attn<4>, hipFuncAttributeMaxDynamicSharedMemorySize, attn_lds_bytes<4>());
        (void)hipFuncSetAttribute((const void*)k_attn<2>, hipFuncAttributeMaxDynamicSharedMemorySize, attn_lds_bytes<2>());
    }
    if (g.ng == 8)
        hipLaunchKernelGGL(k_attn<8>, dim3(blocks), dim3(256), multi ? attn_lds_bytes<8>() : 8 * 256 * 2 * 4, st, items, nitems, Qp, kpool, vpool, page_table, g,
                     group, ppw, part, sc.ctr, par, dyn, multi);
    else if (g.ng == 4)
        hipLaunchKernelGGL(k_attn<4>, dim3(blocks), dim3(256), multi ? attn_lds_bytes<4>() : 8 * 256 * 1 * 4, st, items, nitems, Qp, kpool, vpool, page_table, g,
                     group, ppw, part, sc.ctr, par, dyn, multi);
    else
        hipLaunchKernelGGL(k_attn<2>, dim3(blocks), dim3(256), multi ? attn_lds_bytes<2>() : 8 * 256 * 1 * 4, st, items, nitems, Qp, kpool, vpool, page_table, g,
                     group, ppw, part, sc.ctr, par, dyn, multi);
    CHECK_LAUNCH();
}

// Merge the chunk partials of one (job, kv head, m-tile): log-sum-exp over
// chunks, normalise, and write the merged-heads rows as the o_proj operand
// (merge_heads, web/model/kernels.js:1315-1329, is this indexing). Work item
// i's partial sits at part + i*16*(D + 4) (items are built in that order,
// chunk fastest). One wave per row takes the row's max and weighted sum
// across its lanes (a fixed butterfly order, so the bits depend only on the
// job's chunk count); the weights exp2(m_c - M) go to LDS. Then four groups
// of 256 threads each merge a quarter of the chunks (in order, eight chunks'
// loads in flight), one row's 8 columns a thread, and the quarters are added
// in order through LDS.
constexpr int COMBINE_CMAX = 512, COMBINE_SPLIT = 4;
template <int D>
__global__ __launch_bounds__(1024) void k_attn_combine(const JobDev* __restrict__ jobs, const float* __restrict__ part,
                                                       KVGeom g, int nH, int group, int KU, uint4* __restrict__ Xp,
                                                       float* __restrict__ ctx_out,
                                                       const int32_t* __restrict__ wg_job,
                                                       const float* __restrict__ gate) {
    // rows padded by one float: the four rows a wave reads at one chunk fall in
    // different banks; the quarters' halves in separate arrays, 16 B a thread
    __shared__ float wgt[16][COMBINE_CMAX + 1];
    __shared__ float Ls[16];
    __shared__ float4 red[COMBINE_SPLIT - 1][2][256];
    const int job = wg_job[3 * blockIdx.x], kvh = wg_job[3 * blockIdx.x + 1], mt = wg_job[3 * blockIdx.x + 2];
    const JobDev jb = jobs[job];
    constexpr int W = D + 4;
    const int R = jb.n * group;
    const int nc = jb.nchunk;
    const size_t pstride = (size_t)16 * W;
    const float* base = part + (size_t)(jb.item0 + (kvh * jb.mtq + mt) * nc) * pstride;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    // 16 rows x D columns, 8 a thread, in chunks of at most 128 columns (one
    // chunk up to D = 128, two at D = 256); every thread reaches every barrier
    const int sub = threadIdx.x >> 8, t = threadIdx.x & 255;
    constexpr int CW = D < 128 ? D : 128, PRE = D > 128 ? 4 : 8;   // 8 at D = 256 spills at 128 VGPRs
    const int rl2 = t / (CW / 8);
    const bool live = rl2 < 16 && mt * 16 + rl2 < R;
    const int ca = (sub * nc) / COMBINE_SPLIT, c1 = ((sub + 1) * nc) / COMBINE_SPLIT;
    // the first PRE chunks' values of the first column chunk, loaded before
    // the weights are formed (they do not depend on them)
    float4 pa[PRE], pb[PRE];
    if (live) {
        const float* src = base + (size_t)rl2 * W + 4 + (t % (CW / 8)) * 8;
#pragma unroll
        for (int u = 0; u < PRE; u++)
            if (ca + u < c1) {
                pa[u] = *(const float4*)(src + (ca + u) * pstride);
                pb[u] = *(const float4*)(src + (ca + u) * pstride + 4);
            }
    }
    // only the m-tile's query rows rho < R were written (k_attn skips the rest)
    if (mt * 16 + wave < R) {
        const int rl = wave;   // 16 waves, one row each
        // (max, sum) of chunk `lane` loaded once; chunks past 64 in a loop
        const float2 ml0 = lane < nc ? *(const float2*)(base + lane * pstride + rl * W)
                                     : make_float2(-INFINITY, 0.0f);
        float mloc = ml0.x;
        for (int c = lane + 64; c < nc; c += 64) mloc = fmaxf(mloc, base[c * pstride + rl * W]);
        const float M = wave_max(mloc);
        float lloc = 0.0f;
        if (lane < nc) {
            const float w = ml0.x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml0.x - M);
            wgt[rl][lane] = w;
            lloc += ml0.y * w;
        }
        for (int c = lane + 64; c < nc; c += 64) {
            const float2 ml = *(const float2*)(base + c * pstride + rl * W);
            const float w = ml.x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml.x - M);
            wgt[rl][c] = w;
            lloc += ml.y * w;
        }
        const float L = wave_sum(lloc);
        if (lane == 0) Ls[rl] = L;
    }
    __syncthreads();
    const int rl = rl2;
    const int rho = mt * 16 + rl;
    for (int c0 = 0; c0 < D; c0 += CW) {
        const int d0 = c0 + (t % (CW / 8)) * 8;
        float O[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        if (live) {
            const float* src = base + (size_t)rl * W + 4 + d0;
            auto add = [&](const float4& a, const float4& b, float w) {
                O[0] += a.x * w; O[1] += a.y * w; O[2] += a.z * w; O[3] += a.w * w;
                O[4] += b.x * w; O[5] += b.y * w; O[6] += b.z * w; O[7] += b.w * w;
            };
            int c = ca;
            if (c0 == 0) {
#pragma unroll
                for (int u = 0; u < PRE; u++)
                    if (ca + u < c1) add(pa[u], pb[u], wgt[rl][ca + u]);
                c = ca + PRE < c1 ? ca + PRE : c1;
            }
            for (; c + 8 <= c1; c += 8) {
                float4 a[8], b[8];
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    a[u] = *(const float4*)(src + (c + u) * pstride);
                    b[u] = *(const float4*)(src + (c + u) * pstride + 4);
                }
#pragma unroll
                for (int u = 0; u < 8; u++) add(a[u], b[u], wgt[rl][c + u]);
            }
            for (; c < c1; c++) add(*(const float4*)(src + c * pstride), *(const float4*)(src + c * pstride + 4), wgt[rl][c]);
            if (sub > 0) {
                red[sub - 1][0][t] = make_float4(O[0], O[1], O[2], O[3]);
                red[sub - 1][1][t] = make_float4(O[4], O[5], O[6], O[7]);
            }
        }
        __syncthreads();
        if (sub == 0 && live) {
#pragma unroll
            for (int q = 0; q < COMBINE_SPLIT - 1; q++) {
                const float4 a = red[q][0][t], b = red[q][1][t];
                O[0] += a.x; O[1] += a.y; O[2] += a.z; O[3] += a.w;
                O[4] += b.x; O[5] += b.y; O[6] += b.z; O[7] += b.w;
            }
            float v[8];
            const float L = Ls[rl];
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = O[j] / L;
            const int i = rho / group, gi = rho % group;
            const int r = jb.row0 + i;
            const int k = (kvh * group + gi) * D + d0;
            if (gate) {
                // sigmoid_mul (kernels.js:1822-1839): s = 1/(1+exp(-gate)), s*a
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const float sg = 1.0f / (1.0f + expf(-gate[(size_t)r * nH * D + k + j]));
                    v[j] = sg * v[j];
                }
            }
            if (ctx_out) {
#pragma unroll
                for (int j = 0; j < 8; j++) ctx_out[(size_t)r * nH * D + k + j] = v[j];
            }
            write_hilo(Xp, r, k / 8, KU, v);
        }
        if (c0 + CW < D) __syncthreads();   // `red` is reused by the next chunk
    }
}

void launch_attn_combine(hipStream_t st, const JobDev* jobs, const float* part, const KVGeom& g, int nH, int group,
                         int KU, uint4* Xp, float* ctx_out, const int32_t* wg_job, int nwg, const float* gate) {
    if (nwg <= 0) return;
    if (g.D == 256)
        hipLaunchKernelGGL(k_attn_combine<256>, dim3(nwg), dim3(1024), 0, st, jobs, part, g, nH, group, KU, Xp, ctx_out,
                           wg_job, gate);
    else if (g.D == 128)
        hipLaunchKernelGGL(k_attn_combine<128>, dim3(nwg), dim3(1024), 0, st, jobs, part, g, nH, group, KU, Xp, ctx_out,
                           wg_job, gate);
    else
        hipLaunchKernelGGL(k_attn_combine<64>, dim3(nwg), dim3(1024), 0, st, jobs, part, g, nH, group, KU, Xp, ctx_out,
                           wg_job, gate);
    CHECK_LAUNCH();
}

// k_attn_combine's 64 columns of row m from 64 * unit, by one wave, for at
// most 64 chunks: lane c forms chunk c's weight, lanes 16 q .. 16 q + 15 merge
// quarter q's chunks, 4 columns each, and the first 16 add the quarters in
// order. The result is in lanes 0 .. 15 (columns 4 lane ..). The same values
// by the same operations as k_attn_combine's.
__device__ static inline void combine4(const LxPro& p, int K, int m, int unit, int lane, float (&v)[4]) {
    const int k0 = 64 * unit, h = k0 / p.D, kvh = h / p.group;
    const JobDev jb = p.jobs[p.row_job[m]];
    const int rho = (m - jb.row0) * p.group + h % p.group, W = p.D + 4, nc = jb.nchunk;
    const size_t pstride = (size_t)16 * W;
    const float* base = p.part + (size_t)(jb.item0 + (kvh * jb.mtq + (rho >> 4)) * nc) * pstride + (rho & 15) * W;
    const int sub = lane >> 4;
    const float* src = base + 4 + k0 % p.D + 4 * (lane & 15);
    const int ca = (sub * nc) / COMBINE_SPLIT, c1 = ((sub + 1) * nc) / COMBINE_SPLIT;
    const int most = (nc + COMBINE_SPLIT - 1) / COMBINE_SPLIT;   // chunks of the longest quarter
    float4 x[8];
    auto load = [&](int c0) {
#pragma unroll
        for (int u = 0; u < 8; u++) x[u] = c0 + u < c1 ? *(const float4*)(src + (c0 + u) * pstride) : float4{0, 0, 0, 0};
    };
    load(ca);
    const float2 ml = lane < nc ? *(const float2*)(base + lane * pstride) : make_float2(-INFINITY, 0.0f);
    const float M = wave_max(ml.x);
    const float w = ml.x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml.x - M);
    float lloc = 0.0f;
    if (lane < nc) lloc += ml.y * w;
    const float L = wave_sum(lloc);
    float O[4] = {0, 0, 0, 0};
    for (int c = 0; c < most; c += 8) {
        if (c) load(ca + c);
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const float wc = __shfl(w, (ca + c + u) & 63);
            if (ca + c + u < c1) {
                O[0] += x[u].x * wc; O[1] += x[u].y * wc; O[2] += x[u].z * wc; O[3] += x[u].w * wc;
            }
        }
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float a1 = __shfl_down(O[e], 16), a2 = __shfl_down(O[e], 32), a3 = __shfl_down(O[e], 48);
        v[e] = ((O[e] + a1) + a2) + a3;
        v[e] = v[e] / L;
    }
    if (p.gate && lane < 16) {
        const float4 g = *(const float4*)(p.gate + (size_t)m * K + k0 + 4 * lane);
        const float gv[4] = {g.x, g.y, g.z, g.w};
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float sg = 1.0f / (1.0f + expf(-gv[e]));
            v[e] = sg * v[e];
        }
    }
}

// Whether w's matmul at M rows merges attention's chunks itself: a wave forms
// 64 columns of a row at a time, each behind dependent loads (the row's job,
// its partials, the weights), so the workgroup's columns times rows count,
// over its 8 waves. Up to 2 rounds it beats the launch it saves. A block, us
// (rounds in brackets): hidden 576, 1 row 2.9 less (1), 4 rows 2.1 less (1),
// 6 rows 1.4 less (2), 8 rows 0.6 less (2), 9-12 rows 0.9 to 1.4 more (3);
// hidden 4096, 1 row 1.7 less (2), 2 rows 3 more (4). A lane holds one
// chunk's weight: at most 64.
constexpr int LX_ATTN_COLUMNS = 2 * LX_WAVES;
bool gemm_fuses_attn(const QTensor& w, int M, int chunks) {
    const int len = (w.KU + w.P - 1) / w.P;
    return chunks <= 64 && M <= GEMM_FUSE_ROWS && M * len <= LX_ATTN_COLUMNS;
}

void launch_gemm_attn(hipStream_t st, const QTensor& w, const JobDev* jobs, const int32_t* row_job, const float* part,
                      const KVGeom& g, int group, const float* gate, float* out, int M, int ncu) {
    LxPro p;
    p.part = part;
    p.jobs = jobs;
    p.row_job = row_job;
    p.gate = gate;
    p.D = g.D;
    p.group = group;
    if (w.f32s) launch_lx<1, true, LX_PRO_ATTN>(st, w, nullptr, out, M, ncu, p);
    else launch_lx<1, false, LX_PRO_ATTN>(st, w, nullptr, out, M, ncu, p);
    CHECK_LAUNCH();
}

// =============================================================== embedding ===
// gather_embed_nopos_q8 (web/model/kernels.js:895-917) + round_f16 (the
// embedding rows are rounded like a block's output, stage.js:1365-1370).
__global__ void k_embed(const int32_t* __restrict__ ids, int T, int H, const uint8_t* __restrict__ rec, int Nt, int KU, int P,
                        int f32s, float* __restrict__ x, int round, int nrows) {
    const int t = blockIdx.y;
    const int h = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= T || h >= H) return;
    const int v = ids[t];
    if (v < 0 || v >= nrows) {   // a token outside a shorter table (the MTP's draft rows) reads zero
        x[(size_t)t * H + h] = 0.0f;
        return;
    }
    const int tile = v >> 4, u = h >> 6, lane = (v & 15) + 16 * ((h & 31) >> 3);
    const int byte = 8 * ((h & 63) >> 5) + (h & 7);
    const uint8_t* r = rec + lx_record(tile, u, KU, P, Nt);
    const int8_t q = (int8_t)(r[(tile & 1) * 1024 + lane * 16 + byte] ^ 0x80);
    const uint8_t* sp = r + 2048 + (v & 15) * 8 + (tile & 1) * 4;
    const float sc = f32s ? *(const float*)sp : half_value(*(const uint16_t*)(sp + ((h >> 5) & 1) * 2));
    const float e = (float)q * sc;
    x[(size_t)t * H + h] = round ? round_f16_value(e) : e;
}

void launch_embed(hipStream_t st, const int32_t* ids, int T, const QTensor& wte, float* x, int round) {
    dim3 grid((wte.K + 255) / 256, T);
    hipLaunchKernelGGL(k_embed, grid, dim3(256), 0, st, ids, T, wte.K, wte.codes, wte.Nt, wte.KU, wte.P, wte.f32s, x,
                       round, wte.N);
    CHECK_LAUNCH();
}

// rows[r] = src[r] >= 0 ? x row src[r] : alt row (-1 - src[r]), H floats each:
// the MTP's hidden rows, the session's kept row first (stage.js:1408-1417).
__global__ void k_gather_rows(const float* __restrict__ x, const float* __restrict__ alt,
                              const int32_t* __restrict__ src, int T, int H, float* __restrict__ rows) {
    const int r = blockIdx.y;
    const int h = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= T || h >= H) return;
    const int s = src[r];
    rows[(size_t)r * H + h] = s >= 0 ? x[(size_t)s * H + h] : alt[(size_t)(-1 - s) * H + h];
}

void launch_gather_rows(hipStream_t st, const float* x, const float* alt, const int32_t* src, int T, int H,
                        float* rows) {
    if (T <= 0) return;
    hipLaunchKernelGGL(k_gather_rows, dim3((H + 255) / 256, T), dim3(256), 0, st, x, alt, src, T, H, rows);
    CHECK_LAUNCH();
}

// ==================================================================== top-k ===
// topk_stage / topkRows (web/model/kernels.js:1453-1507, :2129-2144): per row
// the best M (value, index) pairs, larger value first, ties to the lower
// index. Keys pack (order-preserving value bits, ~index), so the order of the
// 64-bit keys is that order and no two are equal; 0 is no key. A workgroup
// takes 4096 keys, 16 a thread, and keeps their best M in order, stage after
// stage until one workgroup's output is left, which writes the pairs.
__device__ static inline uint64_t topk_key(float v, uint32_t i) {
    uint32_t b = f2u(v);
    b = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
    return ((uint64_t)b << 32) | (uint64_t)(0xffffffffu - i);
}

constexpr int TOPK_CH = 4096, TOPK_T = 256, TOPK_PER = TOPK_CH / TOPK_T;

// This thread's 16 keys of the row's chunk at `base`, one of each 256 entries:
// from the head's logits, its planes added in order with a plane's 16 loads
// in flight at once, or from a stage's keys, which come as sorted runs of M:
// there the entry is skewed by a step of 37 a run of 256, so that a thread's
// keys have different ranks (at M = 256 they would all have the same one, and
// the largest of the threads would bound the M-th badly). 0 past the end.
__device__ static inline void topk_load(const float* __restrict__ logits, int planes, size_t stride,
                                        const uint64_t* __restrict__ keys_in, int row, int n, int base,
                                        uint64_t (&key)[TOPK_PER]) {
    const int t = threadIdx.x;
    if (!logits) {
#pragma unroll
        for (int j = 0; j < TOPK_PER; j++) {
            const int i = base + j * TOPK_T + ((t + 37 * j) & (TOPK_T - 1));
            key[j] = i < n ? keys_in[(size_t)row * n + i] : 0;
        }
        return;
    }
    const float* p = logits + (size_t)row * n;
    float v[TOPK_PER];
#pragma unroll
    for (int j = 0; j < TOPK_PER; j++) {
        const int i = base + t + j * TOPK_T;
        v[j] = i < n ? p[i] : 0.0f;
    }
    for (int q = 1; q < planes; q++) {
        p += stride;
        float w[TOPK_PER];
#pragma unroll
        for (int j = 0; j < TOPK_PER; j++) {
            const int i = base + t + j * TOPK_T;
            w[j] = i < n ? p[i] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < TOPK_PER; j++) v[j] = v[j] + w[j];
    }
#pragma unroll
    for (int j = 0; j < TOPK_PER; j++) {
        const int i = base + t + j * TOPK_T;
        key[j] = i < n ? topk_key(v[j], (uint32_t)i) : 0;
    }
}

// Pair or key m of a row: the last stage (vals) writes the pair, the others the key.
__device__ static inline void topk_emit(uint64_t k, int row, int groups, int M, int m, uint64_t* __restrict__ out,
                                        float* __restrict__ vals, uint32_t* __restrict__ ids) {
    if (!vals) {
        out[((size_t)row * groups + blockIdx.x) * M + m] = k;
        return;
    }
    uint32_t b = (uint32_t)(k >> 32);
    b = (b & 0x80000000u) ? (b & 0x7fffffffu) : ~b;
    vals[(size_t)row * M + m] = u2f(b);
    ids[(size_t)row * M + m] = 0xffffffffu - (uint32_t)(k & 0xffffffffu);
}

// How many of s[0 .. n) (n a multiple of 8, 16-byte aligned) are larger than
// each of K keys: every thread reads the same keys, a broadcast.
template <int K>
__device__ static inline void topk_larger(const uint64_t* s, int n, const uint64_t (&k)[K], int (&c)[K]) {
#pragma unroll
    for (int i = 0; i < K; i++) c[i] = 0;
    for (int q = 0; q < n; q += 8) {
        ulonglong2 x[4];
#pragma unroll
        for (int e = 0; e < 4; e++) x[e] = *(const ulonglong2*)(s + q + 2 * e);
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int i = 0; i < K; i++) c[i] += (x[e].x > k[i] ? 1 : 0) + (x[e].y > k[i] ? 1 : 0);
    }
}

// The best M of a chunk, by elimination rather than a sort of all 4096 keys:
// the M-th largest of the threads' largest keys is a key that at least M keys
// reach, and few others do (M = 40: about 45 keys of 4096 in random order;
// above 64 each thread gives the largest of each of its two halves, which
// keeps that bound tight: about 350 at M = 256). Those that reach it are
// gathered and ordered: up to 512 by counting, for each, the larger ones
// (no barriers), more (an unlucky order of the input) by a bitonic sort of
// the next power of two. What bounds it is reading the planes: at 32 rows of
// 151936 logits in 4 planes (78 MB), M = 40, the two stages took 536 us as a
// bitonic sort of every chunk and take 31 now; at 128 rows, M = 256, one
// plane, the three take 204 us (1 row: 68).
__global__ __launch_bounds__(TOPK_T) void k_topk_stage(const float* __restrict__ logits, int planes,
                                                       const uint64_t* __restrict__ keys_in, int n, int M,
                                                       uint64_t* __restrict__ out, float* __restrict__ vals,
                                                       uint32_t* __restrict__ ids) {
    __shared__ __align__(16) uint64_t s[TOPK_CH];
    __shared__ __align__(16) uint64_t mx[2 * TOPK_T];
    __shared__ uint64_t s_thr;
    __shared__ int s_cnt;
    const int t = threadIdx.x, row = blockIdx.y, groups = gridDim.x;
    uint64_t key[TOPK_PER];
    topk_load(logits, planes, (size_t)gridDim.y * n, keys_in, row, n, blockIdx.x * TOPK_CH, key);
    uint64_t top[2] = {0, 0};
#pragma unroll
    for (int j = 0; j < TOPK_PER; j++) {
        uint64_t& m = top[j / (TOPK_PER / 2)];
        m = key[j] > m ? key[j] : m;
    }
    const bool halves = M > 64;
    if (!halves) top[0] = top[1] > top[0] ? top[1] : top[0];
    mx[t] = top[0];
    if (halves) mx[TOPK_T + t] = top[1];
    if (t == 0) {
        s_cnt = 0;
        s_thr = 1;   // fewer than M of the largest are keys: every key stays
    }
    __syncthreads();
    const int nm = halves ? 2 * TOPK_T : TOPK_T;
    if (halves) {
        int c[2];
        topk_larger(mx, nm, top, c);
        if (top[0] && c[0] == M - 1) s_thr = top[0];
        if (top[1] && c[1] == M - 1) s_thr = top[1];
    } else {
        const uint64_t k[1] = {top[0]};
        int c[1];
        topk_larger(mx, nm, k, c);
        if (top[0] && c[0] == M - 1) s_thr = top[0];
    }
    __syncthreads();
    const uint64_t thr = s_thr;
#pragma unroll
    for (int j = 0; j < TOPK_PER; j++)
        if (key[j] >= thr) s[atomicAdd(&s_cnt, 1)] = key[j];
    __syncthreads();
    const int C = s_cnt;
    if (C <= 2 * TOPK_T) {
        const int C8 = (C + 7) & ~7;
        if (C + t < C8) s[C + t] = 0;
        __syncthreads();
        auto keep = [&](uint64_t k, int r) {
            if (k && r < M) topk_emit(k, row, groups, M, r, out, vals, ids);
        };
        if (C <= TOPK_T) {
            const uint64_t k[1] = {t < C ? s[t] : 0};
            int c[1];
            topk_larger(s, C8, k, c);
            keep(k[0], c[0]);
        } else {
            const uint64_t k[2] = {s[t], TOPK_T + t < C ? s[TOPK_T + t] : 0};
            int c[2];
            topk_larger(s, C8, k, c);
            keep(k[0], c[0]);
            keep(k[1], c[1]);
        }
        for (int m = C + t; m < M; m += TOPK_T) topk_emit(0, row, groups, M, m, out, vals, ids);
        return;
    }
    int n2 = 4 * TOPK_T;
    while (n2 < C) n2 <<= 1;
    for (int i = C + t; i < n2; i += TOPK_T) s[i] = 0;
    __syncthreads();
    for (int size = 2; size <= n2; size <<= 1)
        for (int st = size >> 1; st > 0; st >>= 1) {
            for (int p = t; p < n2 / 2; p += TOPK_T) {
                const int i = ((p & ~(st - 1)) << 1) | (p & (st - 1)), l = i | st;
                const uint64_t a = s[i], b = s[l];
                if (((i & size) == 0) ? (a < b) : (a > b)) {
                    s[i] = b;
                    s[l] = a;
                }
            }
            __syncthreads();
        }
    for (int m = t; m < M; m += TOPK_T) topk_emit(s[m], row, groups, M, m, out, vals, ids);
}

// M = 1 (greedy, argmax_rows semantics: web/model/kernels.js:1411-1443): the
// largest key of each chunk, then of the chunks' keys.
__global__ __launch_bounds__(TOPK_T) void k_argmax_stage(const float* __restrict__ logits, int planes,
                                                         const uint64_t* __restrict__ keys_in, int n,
                                                         uint64_t* __restrict__ out, float* __restrict__ vals,
                                                         uint32_t* __restrict__ ids) {
    __shared__ uint64_t red[TOPK_T / 64];
    const int t = threadIdx.x, row = blockIdx.y;
    uint64_t key[TOPK_PER];
    topk_load(logits, planes, (size_t)gridDim.y * n, keys_in, row, n, blockIdx.x * TOPK_CH, key);
    uint64_t best = 0;
#pragma unroll
    for (int j = 0; j < TOPK_PER; j++) best = key[j] > best ? key[j] : best;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const uint64_t x = __shfl_xor((unsigned long long)best, o);
        best = x > best ? x : best;
    }
    if ((t & 63) == 0) red[t >> 6] = best;
    __syncthreads();
    if (t == 0) {
#pragma unroll
        for (int w = 1; w < TOPK_T / 64; w++) best = red[w] > best ? red[w] : best;
        topk_emit(best, row, gridDim.x, 1, 0, out, vals, ids);
    }
}

void launch_topk(hipStream_t st, const float* logits, int planes, int rows, int V, int M, uint64_t* a,
                 uint64_t* b, float* vals, uint32_t* ids) {
    int n = V;
    const float* lg = logits;
    const uint64_t* in = nullptr;
    uint64_t* out = a;
    uint64_t* other = b;
    for (;;) {
        const int groups = (n + TOPK_CH - 1) / TOPK_CH;
        const bool last = groups == 1;
        if (M == 1)
            hipLaunchKernelGGL(k_argmax_stage, dim3(groups, rows), dim3(TOPK_T), 0, st, lg, planes, in, n, out,
                               last ? vals : nullptr, last ? ids : nullptr);
        else
            hipLaunchKernelGGL(k_topk_stage, dim3(groups, rows), dim3(TOPK_T), 0, st, lg, planes, in, n, M, out,
                               last ? vals : nullptr, last ? ids : nullptr);
        CHECK_LAUNCH();
        if (last) break;
        lg = nullptr;
        in = out;
        n = groups * M;
        std::swap(out, other);
    }
}

// The staged keys launch_topk needs for (rows, V, M): the first half (`a`,
// stages 1, 3, ...) and the second (`b`, stages 2, 4, ...), in keys.
void topk_stage_keys(int rows, int V, int M, size_t* a_keys, size_t* b_keys) {
    size_t sa = 0, sb = 0;
    int n = V;
    for (bool to_a = true;; to_a = !to_a) {
        const int groups = (n + TOPK_CH - 1) / TOPK_CH;
        const size_t k = (size_t)rows * groups * M;
        if (to_a) sa = std::max(sa, k);
        else sb = std::max(sb, k);
        if (groups == 1) break;
        n = M == 1 ? groups : groups * M;
    }
    *a_keys = sa;
    *b_keys = sb;
}

// Scratch of the allocation-free top-k entry point (cc_topk_noalloc): the
// staged keys, both halves. Each GPU the library runs on holds its own copy
// until the process ends. Every key a stage reads was written by the stage
// before it in the same call, so nothing in it needs clearing between calls.
// In host code `scratch` names a host-side stand-in, never device memory:
// kernels get the per-device address topk_scratch_setup() looks up.
static __device__ __align__(256) uint64_t scratch[TOPK_SCRATCH_KEYS];

hipError_t topk_scratch_setup(int device, uint64_t** out) {
    static std::mutex mu;
    static uint64_t* ptrs[TOPK_SCRATCH_DEVICES] = {};
    if (device < 0 || device >= TOPK_SCRATCH_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(mu);
    if (!ptrs[device]) {
        uint64_t* p = nullptr;
        const hipError_t e = hipGetSymbolAddress((void**)&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        ptrs[device] = p;
    }
    *out = ptrs[device];
    return hipSuccess;
}

// ============================================================ small kernels ===
__global__ void k_round_f16(float* a, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        a[i] = round_f16_value(a[i]);
}

void launch_round_f16(hipStream_t st, float* a, int64_t n) {
    int64_t blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(k_round_f16, dim3((unsigned)blocks), dim3(256), 0, st, a, n);
    CHECK_LAUNCH();
}

__global__ void k_fill(float* p, int64_t n, float v) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

void launch_fill(hipStream_t st, float* p, int64_t n, float v) {
    int64_t blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(k_fill, dim3((unsigned)blocks), dim3(256), 0, st, p, n, v);
    CHECK_LAUNCH();
}

// Page allocation (web/model/model.js:191-202 ensurePages, replayed for every
// job of the pass in job order): plan[4j..4j+3] = slot, owned, new, prefix.
// The host tracks counts (the stack top and each frame's length); the device
// holds the indices. Job j's k-th new page is the stack entry
// top-1-(prefix+k): what sequential pops would return.
__global__ void k_alloc_pages(const int32_t* __restrict__ plan, int njobs, const uint32_t* __restrict__ free_stack,
                              int top, uint32_t* __restrict__ page_table, int max_pages) {
    const int j = blockIdx.x;
    if (j >= njobs) return;
    const int slot = plan[4 * j], owned = plan[4 * j + 1], nw = plan[4 * j + 2], pre = plan[4 * j + 3];
    for (int k = threadIdx.x; k < nw; k += blockDim.x)
        page_table[(size_t)slot * max_pages + owned + k] = free_stack[top - 1 - (pre + k)];
}

void launch_alloc_pages(hipStream_t st, const int32_t* plan, int njobs, const uint32_t* free_stack, int top,
                        uint32_t* page_table, int max_pages) {
    if (njobs <= 0) return;
    hipLaunchKernelGGL(k_alloc_pages, dim3(njobs), dim3(64), 0, st, plan, njobs, free_stack, top, page_table,
                       max_pages);
    CHECK_LAUNCH();
}

// The next pass's ids from this pass's top-M output: column 0 (the greedy
// token) of each sampled row.
__global__ void k_ids_col0(const uint32_t* __restrict__ ids, int rows, int stride, int32_t* __restrict__ out) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < rows) out[r] = (int32_t)ids[(size_t)r * stride];
}

void launch_ids_col0(hipStream_t st, const uint32_t* ids, int rows, int stride, int32_t* out) {
    if (rows <= 0) return;
    hipLaunchKernelGGL(k_ids_col0, dim3((rows + 255) / 256), dim3(256), 0, st, ids, rows, stride, out);
    CHECK_LAUNCH();
}

// ================================================================ packing ===
// Per-job counts, their prefix sums in job order, then every job's tables. A
// job of n rows at past p needs ceil(n*group/16)
// Q m-tiles, ceil(ceil((p+n)/64)/ppw) chunks of pages per (kv head, m-tile),
// one combine triple per (kv head, m-tile), and nKV*mtq*ng*128 Q-operand
// units; each work item's softmax partial takes 16*(D+4) floats, at the
// item's index in (job, kv head, m-tile, chunk) order. The item list itself
// holds the jobs of several m-tiles first, each (kv head, chunk) as blocks of
// four m-tiles (padded with mt = -1), so one workgroup's four waves read the
// same pages together and the pages come from HBM once; then the jobs of
// one m-tile: first every chunk of ppw pages, then the last, shorter chunks,
// so the blocks a launch hands out last are the short ones (k_attn).
//
// Every workgroup forms the counts and all their prefix sums for itself (four
// jobs a thread, the eight sums together through one wave scan and one
// exchange between the waves, so two barriers); the waves of all workgroups
// then share the tables out: a job to several waves where there are more
// waves than jobs, else several jobs to a wave. launch_pack takes one
// workgroup per PACK_ITEMS work items (a wave then writes about one item a
// lane). What bounds it is latency: one workgroup with a scan per sum took
// 11.7 us for 12 chats, 15.6 for 32, 36 for 16 verify jobs at 4k-32k tokens;
// now 7.3, 7.4 and 7.8.
constexpr int PACK_THREADS = 256, PACK_WAVES = PACK_THREADS / 64;
constexpr int PACK_ITEMS = 256, PACK_BLOCKS_MAX = 64;
static_assert(PACK_MAX_JOBS <= 4 * PACK_THREADS, "four jobs a thread");

__global__ __launch_bounds__(PACK_THREADS) void k_pack(const PackJob* __restrict__ in, int njobs, int step,
                                                       PackGeom g, JobDev* __restrict__ jobs,
                                                       AttnItem* __restrict__ items, int32_t* __restrict__ row_job,
                                                       int32_t* __restrict__ head_rows, int32_t* __restrict__ cwg) {
    // per job: the sums before it (rows, items, combine triples, Q units, head
    // rows), its place in the item list (and of its short chunks), and its counts
    __shared__ int32_t s_row0[PACK_MAX_JOBS], s_item0[PACK_MAX_JOBS], s_cwg0[PACK_MAX_JOBS],
        s_qp0[PACK_MAX_JOBS], s_head0[PACK_MAX_JOBS], s_mtq[PACK_MAX_JOBS], s_nch[PACK_MAX_JOBS],
        s_pos0[PACK_MAX_JOBS], s_posb[PACK_MAX_JOBS], s_part[PACK_WAVES][8];
    const int t = threadIdx.x, ln = t & 63, wv = t >> 6;
    {
        constexpr int NS = 8;   // rows, items, triples, Q units, head rows, list places: multi, full, short
        int a[4][NS], mtq[4], x[NS];
#pragma unroll
        for (int k = 0; k < NS; k++) x[k] = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int j = 4 * t + i;
            mtq[i] = 0;
#pragma unroll
            for (int k = 0; k < NS; k++) a[i][k] = 0;
            if (j < njobs) {
                const PackJob pj = in[j];
                const int tact = pj.past + step + pj.n, pages = (tact + g.page - 1) / g.page;
                const int nch = (pages + g.ppw - 1) / g.ppw;
                mtq[i] = (pj.n * g.group + 15) / 16;
                const bool multi = mtq[i] > 1;
                a[i][0] = pj.n;
                a[i][1] = g.nKV * mtq[i] * nch;
                a[i][2] = g.nKV * mtq[i];
                a[i][3] = g.nKV * mtq[i] * g.ng * 128;
                a[i][4] = g.head ? pj.sampled : 0;
                a[i][5] = multi ? g.nKV * nch * 4 * ((mtq[i] + 3) / 4) : 0;
                a[i][6] = multi ? 0 : g.nKV * (pages / g.ppw);
                a[i][7] = multi ? 0 : g.nKV * (pages % g.ppw != 0);
                s_mtq[j] = mtq[i];
                s_nch[j] = nch;
            }
#pragma unroll
            for (int k = 0; k < NS; k++) x[k] += a[i][k];
        }
        int run[NS];   // the exclusive prefix of this thread's first job
#pragma unroll
        for (int k = 0; k < NS; k++) run[k] = -x[k];
#pragma unroll
        for (int o = 1; o < 64; o <<= 1)
#pragma unroll
            for (int k = 0; k < NS; k++) {
                const int y = __shfl_up(x[k], o);
                if (ln >= o) x[k] += y;
            }
        if (ln == 63)
#pragma unroll
            for (int k = 0; k < NS; k++) s_part[wv][k] = x[k];
        __syncthreads();
        int tot_multi = 0, tot_full = 0;
#pragma unroll
        for (int w = 0; w < PACK_WAVES; w++) {
            tot_multi += s_part[w][5];
            tot_full += s_part[w][6];
#pragma unroll
            for (int k = 0; k < NS; k++) run[k] += w < wv ? s_part[w][k] : 0;
        }
#pragma unroll
        for (int k = 0; k < NS; k++) run[k] += x[k];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int j = 4 * t + i;
            if (j < njobs) {
                s_row0[j] = run[0];
                s_item0[j] = run[1];
                s_cwg0[j] = run[2];
                s_qp0[j] = run[3];
                s_head0[j] = run[4];
                s_pos0[j] = mtq[i] > 1 ? run[5] : tot_multi + run[6];
                s_posb[j] = tot_multi + tot_full + run[7];
            }
#pragma unroll
            for (int k = 0; k < NS; k++) run[k] += a[i][k];
        }
        __syncthreads();
    }
    const int part = 16 * (g.D + 4);
    // waves in groups of wpj (1 when there are at least as many jobs as waves); a group takes every ngr-th job
    const int nw = gridDim.x * PACK_WAVES, wpj = nw > njobs ? nw / njobs : 1, ngr = nw / wpj;
    const int gw = blockIdx.x * PACK_WAVES + wv, sub = gw % wpj;
    if (gw >= ngr * wpj) return;
    const int x0 = sub * 64 + ln, dx = wpj * 64;
    for (int j = gw / wpj; j < njobs; j += ngr) {
        const PackJob pj = in[j];
        const int past = pj.past + step, mtq = s_mtq[j], nch = s_nch[j];
        if (x0 == 0) {
            JobDev jd;
            jd.slot = pj.slot;
            jd.past = past;
            jd.n = pj.n;
            jd.row0 = s_row0[j];
            jd.qp_off = s_qp0[j];
            jd.mtq = mtq;
            jd.item0 = s_item0[j];
            jd.nchunk = nch;
            jd.snap = pj.snap;
            jd.keep = pj.keep;
            jobs[j] = jd;
        }
        if (mtq == 1) {
            const int nfull = ((past + pj.n + g.page - 1) / g.page) / g.ppw;
            for (int x = x0; x < g.nKV * nch; x += dx) {
                const int c = x % nch, h = x / nch;
                const int idx = s_item0[j] + x;   // (kv head, m-tile 0, chunk)
                items[c < nfull ? s_pos0[j] + h * nfull + c : s_posb[j] + h] =
                    AttnItem{pj.slot, past, pj.n, 0, s_qp0[j] + (h * g.ng) * 128, idx * part, h, c * g.ppw};
            }
        } else {
            // (kv head, chunk, block of 4 m-tiles, m-tile): a block is one workgroup
            const int nb = (mtq + 3) / 4, nit = g.nKV * nch * nb * 4;
            for (int x = x0; x < nit; x += dx) {
                const int q = x % 4, b = (x / 4) % nb, c = (x / (4 * nb)) % nch, h = x / (4 * nb * nch);
                const int mt = 4 * b + q;
                if (mt >= mtq) {
                    items[s_pos0[j] + x] = AttnItem{0, 0, 0, -1, 0, 0, 0, 0};
                    continue;
                }
                const int hm = h * mtq + mt;
                const int idx = s_item0[j] + hm * nch + c;
                items[s_pos0[j] + x] =
                    AttnItem{pj.slot, past, pj.n, mt, s_qp0[j] + (hm * g.ng) * 128, idx * part, h, c * g.ppw};
            }
        }
        for (int x = x0; x < g.nKV * mtq; x += dx) {
            const int at = 3 * (s_cwg0[j] + x);
            cwg[at] = j;
            cwg[at + 1] = x / mtq;
            cwg[at + 2] = x % mtq;
        }
        for (int i = x0; i < pj.n; i += dx) row_job[s_row0[j] + i] = j;
        if (g.head)
            for (int i = x0; i < pj.sampled; i += dx)
                head_rows[s_head0[j] + i] = s_row0[j] + pj.n - pj.sampled + i;
    }
}

void launch_pack(hipStream_t st, const PackJob* in, int njobs, int nlaunch, int step, const PackGeom& g, JobDev* jobs,
                 AttnItem* items, int32_t* row_job, int32_t* head_rows, int32_t* cwg) {
    if (njobs <= 0 || njobs > PACK_MAX_JOBS) return;
    const int blocks = std::max(1, std::min(PACK_BLOCKS_MAX, (nlaunch + PACK_ITEMS - 1) / PACK_ITEMS));
    hipLaunchKernelGGL(k_pack, dim3(blocks), dim3(PACK_THREADS), 0, st, in, njobs, step, g, jobs, items, row_job,
                       head_rows, cwg);
    CHECK_LAUNCH();
}

// freePages (web/model/model.js:204-211): push the frame's pages back, last
// owned first, so the next pop returns its first page.
__global__ void k_release_pages(int slot, int owned, uint32_t* __restrict__ free_stack, int top,
                                const uint32_t* __restrict__ page_table, int max_pages) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < owned; i += gridDim.x * blockDim.x)
        free_stack[top + i] = page_table[(size_t)slot * max_pages + owned - 1 - i];
}

void launch_release_pages(hipStream_t st, int slot, int owned, uint32_t* free_stack, int top,
                          const uint32_t* page_table, int max_pages) {
    if (owned <= 0) return;
    hipLaunchKernelGGL(k_release_pages, dim3((owned + 255) / 256), dim3(256), 0, st, slot, owned, free_stack,
                       top, page_table, max_pages);
    CHECK_LAUNCH();
}

// ================================================================ synthetic ===
// A q8 tensor [N, K] generated straight into the tiled layout at row tile
// `row_tile0` of w (fused tensors stack their row tiles). Codes
// clamp(round(N(0,40)), ±127) from the Irwin-Hall generator at index n*K + k;
// f16 scales ~U(1e-4, 4e-4) at index n*ng + g in stream ^ 0x5ca1e.
__global__ void k_gen_q8(uint8_t* __restrict__ rec, int Nt, int KU, int P, int row_tile0, int N, int K,
                         uint64_t seed, uint64_t stream) {
    const int tiles = (N + 15) / 16;
    const int64_t total = (int64_t)tiles * KU * 64;
    const int ng = (K + 31) / 32;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int lane = (int)(i & 63);
        const int64_t tu = i >> 6;
        const int u = (int)(tu % KU), t = (int)(tu / KU);
        const int n = 16 * t + (lane & 15);
        const int tg = row_tile0 + t;
        uint8_t* r = rec + lx_record(tg, u, KU, P, Nt);
        uint8_t b[16];
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const int k = 64 * u + 32 * (j >> 3) + 8 * (lane >> 4) + (j & 7);
            int q = 0;
            if (n < N && k < K) q = gen_code(cc_rng(seed, stream, (uint64_t)n * K + k));
            b[j] = (uint8_t)((q & 0xff) ^ 0x80);
        }
        uint8_t* dst = r + (tg & 1) * 1024 + lane * 16;
#pragma unroll
        for (int j = 0; j < 16; j++) dst[j] = b[j];
        if (lane < 16) {
            for (int h = 0; h < 2; h++) {
                const int gg = 2 * u + h;
                uint16_t sbits = 0;
                if (n < N && gg < ng) sbits = gen_scale_f16(seed, stream ^ 0x5ca1eull, (uint64_t)n * ng + gg, 1e-4, 4e-4);
                *(uint16_t*)(r + 2048 + lane * 8 + (tg & 1) * 4 + h * 2) = sbits;
            }
        }
    }
}

void launch_gen_q8(hipStream_t st, const QTensor& w, int row_tile0, int N, int K, uint64_t seed,
                   uint64_t stream) {
    const int64_t total = (int64_t)((N + 15) / 16) * w.KU * 64;
    int64_t blocks = (total + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(k_gen_q8, dim3((unsigned)blocks), dim3(256), 0, st, w.codes, w.Nt, w.KU, w.P, row_tile0,
                       N, K, seed, stream);
    CHECK_LAUNCH();
}

// Host int8 [N, K] codes + scales -> records: f16 scales [N, ceil(K/32)]
// (f32s = 0), or f32 scales [N, KU], one per 64-wide unit (f32s = 1).
__global__ void k_tile_q8(const int8_t* __restrict__ src, const void* __restrict__ scv, int N, int K,
                          uint8_t* __restrict__ rec, int Nt, int KU, int P, int row_tile0, int f32s) {
    const int tiles = (N + 15) / 16;
    const int64_t total = (int64_t)tiles * KU * 64;
    const int ng = (K + 31) / 32;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int lane = (int)(i & 63);
        const int64_t tu = i >> 6;
        const int u = (int)(tu % KU), t = (int)(tu / KU);
        const int n = 16 * t + (lane & 15);
        const int tg = row_tile0 + t;
        uint8_t* r = rec + lx_record(tg, u, KU, P, Nt);
        uint8_t* dst = r + (tg & 1) * 1024 + lane * 16;
        for (int j = 0; j < 16; j++) {
            const int k = 64 * u + 32 * (j >> 3) + 8 * (lane >> 4) + (j & 7);
            const int q = (n < N && k < K) ? src[(size_t)n * K + k] : 0;
            dst[j] = (uint8_t)((q & 0xff) ^ 0x80);
        }
        if (lane < 16 && f32s) {
            const float* sc = (const float*)scv;
            *(float*)(r + 2048 + lane * 8 + (tg & 1) * 4) = n < N ? sc[(size_t)n * KU + u] : 0.0f;
        } else if (lane < 16) {
            const uint16_t* sc = (const uint16_t*)scv;
            for (int h = 0; h < 2; h++) {
                const int gg = 2 * u + h;
                *(uint16_t*)(r + 2048 + lane * 8 + (tg & 1) * 4 + h * 2) =
                    (n < N && gg < ng) ? sc[(size_t)n * ng + gg] : (uint16_t)0;
            }
        }
    }
}

void launch_tile_q8(hipStream_t st, const int8_t* codes, const void* scales, int N, int K, const QTensor& w,
                    int row_tile0) {
    const int64_t total = (int64_t)((N + 15) / 16) * w.KU * 64;
    int64_t blocks = (total + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(k_tile_q8, dim3((unsigned)blocks), dim3(256), 0, st, codes, scales, N, K, w.codes, w.Nt,
                       w.KU, w.P, row_tile0, w.f32s);
    CHECK_LAUNCH();
}

// Random KV rows 0..tokens-1 of a slot in one layer's pool (which: 0 = K,
// 1 = V): the generator of the test oracle (codes uniform in ±127 at index
// base*D + d, base = ((key << 24) + t)*nKV + head; one f16 scale
// ~U(0.005, 0.02) at base, replicated into every 32-block).
__global__ void k_fill_kv(uint8_t* __restrict__ pool, const uint32_t* __restrict__ page_table, int slot,
                          int tokens, KVGeom g, uint64_t seed, uint64_t stream, uint64_t key, int which) {
    const int D = g.D;
    const int64_t total = (int64_t)tokens * g.nKV * D;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int d = (int)(i % D);
        const int64_t tn = i / D;
        const int n = (int)(tn % g.nKV), t = (int)(tn / g.nKV);
        const uint64_t base = ((key << 24) + (uint64_t)t) * (uint64_t)g.nKV + (uint64_t)n;
        const uint64_t r = cc_rng(seed, stream, base * (uint64_t)D + (uint64_t)d);
        const int8_t code = (int8_t)((int)((r >> 8) % 255u) - 127);
        const uint32_t page = page_table[(size_t)slot * g.max_pages + t / g.page];
        const int s = t % g.page;
        uint8_t* blk = pool + ((size_t)page * g.nKV + n) * g.blk;
        const uint8_t biased = (uint8_t)((uint8_t)code ^ 0x80u);
        if (which == 0) blk[(size_t)s * D + kpos(d, D)] = biased;
        else blk[vcode_at(d, s, D)] = biased;
        if ((d & 31) == 0) {
            const float sc = half_value(gen_scale_f16(seed, stream ^ 0x5ca1eull, base, 0.005, 0.02));
            const int b = d >> 5;
            if (which == 0) *(float*)(blk + 64 * D + ((size_t)s * g.ng + b) * 4) = sc;
            else *(float*)(blk + 64 * D + (size_t)vscale_at(b, s, g.ng) * 4) = sc;
        }
    }
}

void launch_fill_kv(hipStream_t st, uint8_t* pool, const uint32_t* page_table, int slot, int tokens,
                    const KVGeom& g, uint64_t seed, uint64_t stream, uint64_t key, int which) {
    const int64_t total = (int64_t)tokens * g.nKV * g.D;
    if (total <= 0) return;
    int64_t blocks = (total + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(k_fill_kv, dim3((unsigned)blocks), dim3(256), 0, st, pool, page_table, slot, tokens, g,
                       seed, stream, key, which);
    CHECK_LAUNCH();
}

// Device block layout <-> the reference's rows (kernels.js:999-1022): row
// word w < D/4 packs codes 4w..4w+3 (low byte first, signed: the pool's
// biased bytes ^ 0x80); then D/32 f32 scales.
__global__ void k_kv_ref(uint8_t* __restrict__ pool, const uint32_t* __restrict__ page_table, int slot, int head,
                         int t0, int t1, KVGeom g, int which, uint32_t* __restrict__ rows, int to_ref) {
    const int D = g.D, RW = D / 4 + g.ng;
    const int64_t total = (int64_t)(t1 - t0) * RW;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int w = (int)(i % RW), t = t0 + (int)(i / RW);
        const uint32_t page = page_table[(size_t)slot * g.max_pages + t / g.page];
        const int s = t % g.page;
        uint8_t* blk = pool + ((size_t)page * g.nKV + head) * g.blk;
        if (w < D / 4) {
            uint8_t* p[4];
            for (int j = 0; j < 4; j++) {
                const int d = 4 * w + j;
                p[j] = which == 0 ? blk + (size_t)s * D + kpos(d, D) : blk + vcode_at(d, s, D);
            }
            if (to_ref) {
                uint32_t word = 0;
                for (int j = 0; j < 4; j++) word |= (uint32_t)(*p[j] ^ 0x80u) << (8 * j);
                rows[i] = word;
            } else {
                const uint32_t word = rows[i];
                for (int j = 0; j < 4; j++) *p[j] = (uint8_t)((word >> (8 * j)) ^ 0x80u);
            }
        } else {
            const int b = w - D / 4;
            uint32_t* sp = which == 0 ? (uint32_t*)(blk + 64 * D + ((size_t)s * g.ng + b) * 4)
                                      : (uint32_t*)(blk + 64 * D + (size_t)vscale_at(b, s, g.ng) * 4);
            if (to_ref) rows[i] = *sp;
            else *sp = rows[i];
        }
    }
}

void launch_kv_to_ref(hipStream_t st, const uint8_t* pool, const uint32_t* page_table, int slot, int head, int t0,
                      int t1, const KVGeom& g, int which, uint32_t* out) {
    const int64_t total = (int64_t)(t1 - t0) * (g.D / 4 + g.ng);
    if (total <= 0) return;
    hipLaunchKernelGGL(k_kv_ref, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, (uint8_t*)pool,
                       page_table, slot, head, t0, t1, g, which, out, 1);
    CHECK_LAUNCH();
}

void launch_kv_from_ref(hipStream_t st, uint8_t* pool, const uint32_t* page_table, int slot, int head, int t0,
                        int t1, const KVGeom& g, int which, const uint32_t* in) {
    const int64_t total = (int64_t)(t1 - t0) * (g.D / 4 + g.ng);
    if (total <= 0) return;
    hipLaunchKernelGGL(k_kv_ref, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, pool, page_table, slot,
                       head, t0, t1, g, which, (uint32_t*)in, 0);
    CHECK_LAUNCH();
}

// Sum the K splits of a projection: out[m][n] = sum_s part[s][m][n], in order.
__global__ void k_sum_splits(const float* __restrict__ part, int splits, int M, int N, float* __restrict__ out) {
    const int64_t total = (int64_t)M * N;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        float p = part[i];
        for (int s = 1; s < splits; s++) p = p + part[(size_t)s * total + i];
        out[i] = p;
    }
}

void launch_sum_splits(hipStream_t st, const float* part, int splits, int M, int N, float* out) {
    const int64_t total = (int64_t)M * N;
    int64_t blocks = (total + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(k_sum_splits, dim3((unsigned)blocks), dim3(256), 0, st, part, splits, M, N, out);
    CHECK_LAUNCH();
}

// ------------------------------------------------ to and from the host ---
// A pass's small tables, its f16 rows and its results cross the link inside
// kernels that read or write the context's pinned host memory 16 bytes a
// thread, each byte once: a copy on its own waits for the copy engine and
// hands over between queues, about 10 us each way, which a pass of one block
// (150 us of kernels) pays twice.
__global__ void k_copy16(const uint4* __restrict__ src, uint4* __restrict__ dst, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

void launch_copy16(hipStream_t st, const void* src, void* dst, size_t bytes) {
    const int64_t n = (int64_t)((bytes + 15) / 16);
    if (n <= 0) return;
    hipLaunchKernelGGL(k_copy16, dim3((unsigned)std::min<int64_t>((n + 255) / 256, 65536)), dim3(256), 0, st,
                       (const uint4*)src, (uint4*)dst, n);
    CHECK_LAUNCH();
}

// The f16 rows a pass past position 0 is handed, as f32, 8 values a thread.
__global__ void k_rows_in(const uint4* __restrict__ hidden, int64_t n8, float4* __restrict__ x) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n8; i += (int64_t)gridDim.x * blockDim.x) {
        const uint4 q = hidden[i];
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = half_value((uint16_t)(w[e >> 1] >> (16 * (e & 1))));
        x[2 * i] = make_float4(v[0], v[1], v[2], v[3]);
        x[2 * i + 1] = make_float4(v[4], v[5], v[6], v[7]);
    }
}

void launch_rows_in(hipStream_t st, const uint16_t* hidden, int64_t n, float* x) {
    if (n <= 0) return;
    const int64_t n8 = n / 8;
    hipLaunchKernelGGL(k_rows_in, dim3((unsigned)std::min<int64_t>((n8 + 255) / 256, 65536)), dim3(256), 0, st,
                       (const uint4*)hidden, n8, (float4*)x);
    CHECK_LAUNCH();
}

// Rows of f16 values kept as f32 -> their half bits (exact), 8 values a thread.
__global__ void k_to_half_bits(const float4* __restrict__ x, int64_t n8, uint4* __restrict__ out) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n8; i += (int64_t)gridDim.x * blockDim.x) {
        const float4 a = x[2 * i], b = x[2 * i + 1];
        out[i] = make_uint4(half_bits(a.x) | (uint32_t)half_bits(a.y) << 16, half_bits(a.z) | (uint32_t)half_bits(a.w) << 16,
                            half_bits(b.x) | (uint32_t)half_bits(b.y) << 16, half_bits(b.z) | (uint32_t)half_bits(b.w) << 16);
    }
}

void launch_to_half_bits(hipStream_t st, const float* x, int64_t n, uint16_t* out) {
    if (n <= 0) return;
    const int64_t n8 = n / 8;
    hipLaunchKernelGGL(k_to_half_bits, dim3((unsigned)std::min<int64_t>((n8 + 255) / 256, 65536)), dim3(256), 0, st,
                       (const float4*)x, n8, (uint4*)out);
    CHECK_LAUNCH();
}
