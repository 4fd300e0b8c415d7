// Grouped G256 projection for small row counts (decode GEMV path).
//
// Arithmetic: routed_storage_n32_consumer.cpp:124-161 (projection_n32_job) and
// dense_g256_consumer.cpp:116-143 (compact_projection): per output column an
// exact integer dot per 256-group, then the fp32 group tree in ascending
// group order.  The dot uses v_dot4_i32_i8 on the int8 activation layout and
// codes split into even/odd bytes (common.hpp).
//
// Work split: one block (4 waves) owns one segment (one weight bank and its
// routes) and NT consecutive 32-column tiles.  The block stages the code
// blocks of GC groups (NT*GC <= 8 blocks of 4 KiB) into LDS with 128-bit
// coalesced loads, then every thread computes one (tile, group, column)
// integer dot for each route; the group tree runs in a second pass.
#include "kernels.hpp"
#include "timing.hpp"
#include "act.hpp"

namespace ornith {

constexpr int kPad = 1056;          // LDS words per (tile, group) block: 32x32 + 32 (bank spread)
constexpr int kRouteBatch = 16;     // routes whose running sums are kept in LDS

template <int TILE, Out MODE>
__global__ __launch_bounds__(256) void project_gemv_kernel(ProjArgs a, int NT, int GC) {
    __shared__ uint32_t lw[8 * kPad];
    __shared__ uint32_t lm[8 * 32];
    __shared__ uint32_t la[8 * 64];
    __shared__ float lsa[8], lss[8];
    __shared__ float lterm[8][32];
    __shared__ float lrun[kRouteBatch][256];
    __shared__ int lrow[kRouteBatch], lroute[kRouteBatch];

    const int tid = threadIdx.x;
    if (a.nseg && int(blockIdx.x) >= *a.nseg) return;
    const Segment sg = a.segments ? a.segments[blockIdx.x] : Segment{0, 0, a.dense_rows, 0};
    const bool shared = sg.bank == kShared;
    const uint32_t* codes = shared ? a.shared_codes : a.codes + size_t(sg.bank) * a.bank_words;
    const uint32_t* meta = shared ? a.shared_meta : a.meta + size_t(sg.bank) * a.bank_meta_words;
    const int GS = a.K / kGroup;
    const int ntiles = (a.N + 31) / 32;
    const int tile0 = blockIdx.y * NT;
    const int pairs = NT * GC * 32;
    const int cols = NT * 32;

    for (int rb = 0; rb < sg.count; rb += kRouteBatch) {
        const int nr = min(kRouteBatch, sg.count - rb);
        if (tid < nr) {
            const int route = a.routes ? a.routes[sg.first + rb + tid] : rb + tid;
            lroute[tid] = route;
            lrow[tid] = a.row_mode == 0 ? route : (route < a.R ? route / kTop : route - a.R);
        }
        for (int g0 = 0; g0 < GS; g0 += GC) {
            const int gc = min(GC, GS - g0);
            __syncthreads();
            // ---- stage code blocks (tile tl, group gl) and metadata ----
            for (int q = tid; q < NT * gc * 256; q += 256) {
                const int blk = q >> 8, within = (q & 255) * 4;     // word offset inside 1024-word block
                const int tl = blk / gc, gl = blk % gc;
                const int t = tile0 + tl, g = g0 + gl;
                uint4 v = make_uint4(0, 0, 0, 0);
                if (t < ntiles) {
                    if (TILE == 32) {
                        v = *reinterpret_cast<const uint4*>(codes + ((size_t(t) * GS + g) * 32) * 32 + within);
                    } else {
                        const int j = within >> 5, n32 = within & 31, h = n32 >> 4, n16 = n32 & 15;
                        if ((2 * t + h) * 16 < a.N)
                            v = *reinterpret_cast<const uint4*>(codes + ((size_t(2 * t + h) * GS + g) * 32 + j) * 16 + n16);
                    }
                }
                *reinterpret_cast<uint4*>(&lw[(tl * gc + gl) * kPad + within]) = v;
            }
            for (int q = tid; q < NT * gc * 32; q += 256) {
                const int blk = q >> 5, n = q & 31, tl = blk / gc, gl = blk % gc;
                const int t = tile0 + tl, g = g0 + gl, col = t * 32 + n;
                uint32_t m = 0;
                if (col < a.N) {
                    if (TILE == 32) m = meta[(size_t(t) * GS + g) * 32 + n];
                    else m = meta[(size_t(col / 16) * GS + g) * 16 + (col & 15)];
                }
                lm[blk * 32 + n] = m;
            }
            for (int r = 0; r < nr; ++r) {
                const int row = lrow[r];
                // ---- stage this route's activation words for the chunk ----
                for (int q = tid; q < gc * 64; q += 256)
                    la[q] = a.act_words[size_t(row) * (a.K / 4) + size_t(g0) * 64 + q];
                if (tid < gc) {
                    const float sa = f16_bits_to_f32(a.act_scales[size_t(row) * GS + g0 + tid]);
                    lsa[tid] = sa;
                    lss[tid] = sa * float(a.act_sums[size_t(row) * GS + g0 + tid]);
                }
                __syncthreads();
                if (tid < NT * gc * 32) {
                    const int blk = tid >> 5, n = tid & 31, gl = blk % gc;
                    const uint32_t* wb = &lw[blk * kPad + n];
                    const uint32_t* ab = &la[gl * 64];
                    int dot = 0;
#pragma unroll 8
                    for (int c = 0; c < 32; ++c) {
                        const uint32_t w = wb[c * 32];
                        dot = dot4(code_even(w), int(ab[2 * c]), dot);
                        dot = dot4(code_odd(w), int(ab[2 * c + 1]), dot);
                    }
                    lterm[blk][n] = tree_term(dot, lsa[gl], lss[gl], lm[blk * 32 + n]);
                }
                __syncthreads();
                if (tid < cols) {
                    const int tl = tid >> 5, n = tid & 31;
                    float v = g0 == 0 ? 0.f : lrun[r][tid];
                    for (int gl = 0; gl < gc; ++gl) v = v + lterm[tl * gc + gl][n];
                    lrun[r][tid] = v;
                }
            }
        }
        __syncthreads();
        // ---- write the finished rows ----
        for (int q = tid; q < nr * cols; q += 256) {
            const int r = q / cols, cidx = q % cols;
            const int col = tile0 * 32 + cidx;
            if (col >= a.N) continue;
            float v = lrun[r][cidx];
            if (MODE == Out::Routed) {
                if (shared) v = bf16_round(v);   // shared linear outputs are bf16 (:226-227)
                a.out[size_t(lroute[r]) * a.N + col] = v;
                if (!isfinite(v)) atomicOr(a.sticky, a.flag_projection);
            } else {
                const size_t o = size_t(lroute[r]) * a.N + col;
                const uint16_t b = f32_to_bf16_bits(v);
                uint32_t f = 0;
                if (!isfinite(v)) f |= a.flag_projection;
                if ((b & 0x7f80u) == 0x7f80u) f |= a.flag_bf16;
                if (a.out) a.out[o] = v;
                if (a.out_bf16) a.out_bf16[o] = b;
                flag_or(a.sticky, f);
            }
        }
        __syncthreads();
    }
}

// Dense weight-streaming projection for up to kDenseStreamRows rows on the
// int8 matrix cores.  One block owns 32 output columns; wave w owns 256-group
// w of the current NW-group pass, so every load of the block is issued before
// its first product and the bank crosses HBM once for any row count.
//  - Codes: load u (0..7) of lane li + 16q takes word j = 4u + q of column li
//    of each 16-column half, so a load of an N16 tile is 256 contiguous bytes
//    (of an N32 tile four 64-byte halves of its rows; the other half's load
//    takes the rest).  v_mfma_i32_16x16x64_i8 s pairs words u = 2s, 2s + 1
//    (unpacked: even codes, odd codes) with activation chunks 8s + q and
//    8s + 4 + q.  Any pairing of K is exact: |dot| < 2^19.
//  - The product is (codes x activations): lane li + 16q ends with columns
//    4q + 0..3 of activation row li, so a row's scale and sum are one value
//    per lane and the four columns' metadata one 16-byte load.
//  - Terms (tree_term) meet in LDS; one thread per (row, column) adds them in
//    ascending group order (the fp32 tree of dense_g256_consumer.cpp:116-143),
//    so results equal project_gemv_kernel's bit for bit.
// FP > 0 (a.dense_x set): the wave also prepares its group of the activations
// from the bf16 input, FP passes of four rows (the recipe of act_bf16_block),
// into LDS while its codes are in flight; every block repeats that work, so it
// is done up to dense_fused_rows rows, and above them the activations come from
// the workspace.
// Bound by latency: the weights of a 6144 x 2048 linear are 1 us of HBM time;
// a call is the kernel boundaries (~1.1 us each), the loads' round trip and the
// two exchanges through LDS.  Graph-timed per call at 6144 x 2048, activation
// launch included, against the v_dot4 kernel before it (rows one after another
// on the VALU): 1 row 5.4 -> 5.0 us, 4 rows 8.0 -> 5.3, 8 rows 12.3 -> 7.2,
// 16 rows 15.7 -> 7.6, 32 rows 23.5 -> 9.4, 64 rows 39.5 -> 12.1; at 2048 x
// 4096 1 row 8.0 -> 6.3, 32 rows 37.8 -> 10.8, 64 rows 69.2 -> 17.7.
typedef int mfma_i32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));   // metadata is 4-byte aligned

template <int TILE, int MT, int FP, int NW>
__global__ __launch_bounds__(64 * NW) void dense_stream_kernel(ProjArgs a) {
    static_assert(FP == 0 || (MT == 1 && FP <= 2), "fused rows fit one row tile");
    constexpr int ROWS = 16 * MT, NT = 64 * NW, OUT = (ROWS * 32 + NT - 1) / NT;
    constexpr int kTermStride = 36;                // floats per row: 16-byte stores spread over the banks
    constexpr int kActStride = 72;                 // words per row: conflict-free 8-byte reads
    // one LDS area per wave: its activation rows (32 at a time), then its terms
    constexpr int kActRows = ROWS < 32 ? ROWS : 32;
    constexpr int kWaveWords = kActRows * kActStride > ROWS * kTermStride ? kActRows * kActStride : ROWS * kTermStride;
    __shared__ __attribute__((aligned(16))) uint32_t s_wave[NW][kWaveWords];
    __shared__ float2 s_scale[FP ? NW : 1][FP ? 16 : 1];

    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, q = lane >> 4;
    const int GS = a.K / kGroup, M = a.dense_rows;
    // a missing second 16-column half (N % 32 == 16) repeats the first; its
    // columns are never written
    const int half1 = 2 * int(blockIdx.x) + 1 < (a.N >> 4) ? 1 : 0;
    float run[OUT];
#pragma unroll
    for (int i = 0; i < OUT; ++i) run[i] = 0.f;
    uint32_t flags = 0;
    uint32_t* s_act = s_wave[w];
    // the wave's own LDS words, written by other lanes of it
    auto wave_fence = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };

    for (int g0 = 0; g0 < GS; g0 += NW) {
        // a wave past the last group reads group GS - 1 and writes no term
        const int g = min(g0 + w, GS - 1);
        const bool gv = g0 + w < GS;
        // ---- inputs (fused), then codes and metadata, then the workspace's activations ----
        uint4 xa[FP ? FP : 1][2];
        if constexpr (FP > 0) {
#pragma unroll
            for (int i = 0; i < FP; ++i) {
                const uint16_t* src = a.dense_x + size_t(min(4 * i + q, M - 1)) * a.K + g * kGroup + quarter_base(li);
                xa[i][0] = *reinterpret_cast<const uint4*>(src);
                xa[i][1] = *reinterpret_cast<const uint4*>(src + 8);
            }
        }
        uint32_t wr[2][8];
        u32x4 mw[2];
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
            const uint32_t* src;
            const uint32_t* msrc;
            if constexpr (TILE == 32) {
                src = a.codes + (size_t(blockIdx.x) * GS + g) * 1024 + 32 * q + 16 * ct + li;
                msrc = a.meta + (size_t(blockIdx.x) * GS + g) * 32 + 16 * ct + 4 * q;
            } else {
                const size_t block = size_t(2 * int(blockIdx.x) + (ct ? half1 : 0)) * GS + g;
                src = a.codes + block * 512 + 16 * q + li;
                msrc = a.meta + block * 16 + 4 * q;
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) wr[ct][u] = load_once(src + u * 4 * TILE);
            mw[ct] = *reinterpret_cast<const u32x4_a4*>(msrc);
        }
        uint2 fa2[MT][8];                          // [row tile][2s + e]: chunk 8s + 4e + q
        float sa[MT], ss[MT];
        if constexpr (FP == 0) {
            // 16 lanes per row, four rows per load; each half of 32 rows
            // passes through LDS into the products' layout (loaded straight
            // in it, 32 bytes of 16 rows per instruction, the call took 17.1
            // instead of 12.1 us at 64 rows, 11.9 instead of 9.4 at 32)
            u32x4 av[ROWS / 4];
#pragma unroll
            for (int i = 0; i < ROWS / 4; ++i)
                av[i] = *reinterpret_cast<const u32x4*>(a.act_words + size_t(min(4 * i + q, M - 1)) * (a.K / 4) +
                                                        g * 64 + 4 * li);
            uint32_t sbits[MT];
            int sum[MT];
#pragma unroll
            for (int rt = 0; rt < MT; ++rt) {
                const int row = min(16 * rt + li, M - 1);
                sbits[rt] = a.act_scales[size_t(row) * GS + g];
                sum[rt] = a.act_sums[size_t(row) * GS + g];
            }
#pragma unroll
            for (int h = 0; h < ROWS / kActRows; ++h) {
                if (h) wave_fence();
#pragma unroll
                for (int i = 0; i < kActRows / 4; ++i)
                    *reinterpret_cast<u32x4*>(&s_act[(4 * i + q) * kActStride + 4 * li]) = av[h * (kActRows / 4) + i];
                wave_fence();
#pragma unroll
                for (int rt = 0; rt < kActRows / 16; ++rt)
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        fa2[h * (kActRows / 16) + rt][u] =
                            *reinterpret_cast<const uint2*>(&s_act[(16 * rt + li) * kActStride + 8 * u + 2 * q]);
            }
#pragma unroll
            for (int rt = 0; rt < MT; ++rt) {
                sa[rt] = f16_bits_to_f32(uint16_t(sbits[rt]));
                ss[rt] = sa[rt] * float(sum[rt]);
            }
        } else {
            // the input's first use stays behind the code loads (its wait
            // would otherwise come before they are issued)
#pragma unroll
            for (int i = 0; i < FP; ++i)
                asm volatile("" : "+v"(xa[i][0].x), "+v"(xa[i][0].y), "+v"(xa[i][0].z), "+v"(xa[i][0].w),
                                  "+v"(xa[i][1].x), "+v"(xa[i][1].y), "+v"(xa[i][1].z), "+v"(xa[i][1].w));
#pragma unroll
            for (int i = 0; i < FP; ++i) {
                const uint32_t u[8] = {xa[i][0].x, xa[i][0].y, xa[i][0].z, xa[i][0].w,
                                       xa[i][1].x, xa[i][1].y, xa[i][1].z, xa[i][1].w};
                float v[16];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    v[2 * e] = bf16_bits_to_f32(u[e] & 0xffffu);
                    v[2 * e + 1] = bf16_bits_to_f32(u[e] >> 16);
                }
                uint32_t f = 0;
#pragma unroll
                for (int e = 0; e < 16; ++e) if (!isfinite(v[e])) f |= a.flag_input;
                h128_quarter(v);
                uint32_t w4[4];
                uint16_t sbits;
                int sum;
                quantize_quarter_fast<127>(v, w4, sbits, sum, f, a.flag_input | a.flag_act, a.flag_act);
                const int row = 4 * i + q;         // rows past M repeat row M - 1
                *reinterpret_cast<uint4*>(&s_act[row * kActStride + quarter_base(li) / 4]) =
                    make_uint4(w4[0], w4[1], w4[2], w4[3]);
                if (li == 0) {
                    const float scale = f16_bits_to_f32(sbits);
                    s_scale[w][row] = make_float2(scale, scale * float(sum));
                }
                flags |= f;
            }
            wave_fence();
            const int row = min(li, min(4 * FP, M) - 1);
#pragma unroll
            for (int u = 0; u < 8; ++u)
                fa2[0][u] = *reinterpret_cast<const uint2*>(&s_act[row * kActStride + 8 * u + 2 * q]);
            const float2 sc = s_scale[w][row];
            sa[0] = sc.x;
            ss[0] = sc.y;
        }
        wave_fence();                              // the terms take the activations' place
        // ---- exact dots and the group's terms ----
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
            mfma_i32x4 acc[MT];
#pragma unroll
            for (int rt = 0; rt < MT; ++rt) acc[rt] = mfma_i32x4{0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const uint32_t w0 = wr[ct][2 * s], w1 = wr[ct][2 * s + 1];
                const mfma_i32x4 fb = {code_even(w0), code_odd(w0), code_even(w1), code_odd(w1)};
#pragma unroll
                for (int rt = 0; rt < MT; ++rt) {
                    const mfma_i32x4 fa = {int(fa2[rt][2 * s].x), int(fa2[rt][2 * s].y), int(fa2[rt][2 * s + 1].x),
                                           int(fa2[rt][2 * s + 1].y)};
                    acc[rt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fb, fa, acc[rt], 0, 0, 0);
                }
            }
            if (gv) {
#pragma unroll
                for (int rt = 0; rt < MT; ++rt) {
                    f32x4 t;
#pragma unroll
                    for (int r = 0; r < 4; ++r) t[r] = tree_term(acc[rt][r], sa[rt], ss[rt], mw[ct][r]);
                    *reinterpret_cast<f32x4*>(&s_wave[w][(16 * rt + li) * kTermStride + 16 * ct + 4 * q]) = t;
                }
            }
        }
        __syncthreads();
        const int gc = min(NW, GS - g0);
#pragma unroll
        for (int i = 0; i < OUT; ++i) {
            const int r = min((tid >> 5) + i * (NT / 32), ROWS - 1), c = tid & 31;
            for (int gl = 0; gl < gc; ++gl) run[i] = run[i] + __uint_as_float(s_wave[gl][r * kTermStride + c]);
        }
        if (g0 + NW < GS) __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < OUT; ++i) {
        const int r = (tid >> 5) + i * (NT / 32), c = 32 * int(blockIdx.x) + (tid & 31);
        if (r >= M || c >= a.N) continue;
        const float v = run[i];
        const size_t o = size_t(r) * a.N + c;
        const uint16_t b = f32_to_bf16_bits(v);
        if (!isfinite(v)) flags |= a.flag_projection;
        if ((b & 0x7f80u) == 0x7f80u) flags |= a.flag_bf16;
        if (a.out) a.out[o] = v;
        if (a.out_bf16) a.out_bf16[o] = b;
    }
    flag_or(a.sticky, flags);
}

// Waves per block: one per 256-group of K up to 16 (8 with 64 rows, whose
// activations take the registers of a 16-wave block), at least 4.
template <int TILE, int MT, int FP> void go_dense_stream(const ProjArgs& a, hipStream_t s) {
    const dim3 grid((a.N + 31) / 32);
    const int GS = a.K / kGroup;
    if (GS <= 4 || FP > 1)                         // eight fused rows: K <= 1024 (dense_fused_rows)
        timed_launch("dense_stream", dense_stream_kernel<TILE, MT, FP, 4>, grid, dim3(256), 0, s, a);
    else if constexpr (FP <= 1) {
        if (GS <= 8 || MT > 2)
            timed_launch("dense_stream", dense_stream_kernel<TILE, MT, FP, 8>, grid, dim3(512), 0, s, a);
        else if constexpr (MT <= 2)
            timed_launch("dense_stream", dense_stream_kernel<TILE, MT, FP, 16>, grid, dim3(1024), 0, s, a);
    }
}

template <int TILE> void launch_dense_stream(const ProjArgs& a, hipStream_t s) {
    const int M = a.dense_rows;
    if (a.dense_x && M <= 4) go_dense_stream<TILE, 1, 1>(a, s);
    else if (a.dense_x) go_dense_stream<TILE, 1, 2>(a, s);
    else if (M <= 16) go_dense_stream<TILE, 1, 0>(a, s);
    else if (M <= 32) go_dense_stream<TILE, 2, 0>(a, s);
    else go_dense_stream<TILE, 4, 0>(a, s);
}

hipError_t launch_project_gemv(const ProjArgs& a, int max_segments, Out mode, hipStream_t s) {
    const int GS = a.K / kGroup;
    const int GC = GS < 8 ? GS : 8;
    const int NT = 8 / GC;
    const int ntiles = (a.N + 31) / 32;
    const dim3 grid(max_segments, (ntiles + NT - 1) / NT);
    if (max_segments <= 0) return hipSuccess;
    if (mode == Out::Dense && !a.segments && a.dense_rows <= kDenseStreamRows) {
        if (a.tile == 32) launch_dense_stream<32>(a, s);
        else launch_dense_stream<16>(a, s);
        return hipGetLastError();
    }
    if (a.tile == 32) {
        if (mode == Out::Routed) timed_launch("dense_gemv", project_gemv_kernel<32, Out::Routed>, dim3(grid), dim3(256), 0, s, a, NT, GC);
        else timed_launch("dense_gemv", project_gemv_kernel<32, Out::Dense>, dim3(grid), dim3(256), 0, s, a, NT, GC);
    } else {
        if (mode == Out::Routed) timed_launch("dense_gemv", project_gemv_kernel<16, Out::Routed>, dim3(grid), dim3(256), 0, s, a, NT, GC);
        else timed_launch("dense_gemv", project_gemv_kernel<16, Out::Dense>, dim3(grid), dim3(256), 0, s, a, NT, GC);
    }
    return hipGetLastError();
}

}  // namespace ornith
