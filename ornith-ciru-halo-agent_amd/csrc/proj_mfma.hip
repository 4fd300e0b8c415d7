// G256 LM head on the int8 matrix cores.
//
// Arithmetic is the reference's A8 math, exactly: per (row, column,
// 256-group) the integer dot sum_k code*q is formed on the int8 matrix cores
// (exact: |dot| < 2^19), then the fp32 group tree
// value = value + (RN(sw*RN(sa*dot)) + RN(off*RN(sa*sum))) runs in ascending
// group order on the VALU (dense_g256_api.h:35-37).
//
// MFMA operand layout of v_mfma_i32_16x16x64_i8 (verified on gfx950): lane
// i+16q supplies the 16 bytes of row/column i for k-group q, A and B bytes
// pair positionally, and output register r of lane l is C[4*(l/16)+r][l%16].
// Both operands use this build's byte order (even codes then odd codes per
// 8-value chunk), so the logical k pairing matches and the integer dot is
// exact.
#include "kernels.hpp"
#include "timing.hpp"
#include "decode.hpp"
#include "mfma.hpp"
#include <algorithm>
#include <utility>

namespace ornith {

constexpr int kMT = 64, kNT = 128;   // rows, columns per block (33..64 rows)

// Top-1 order of numpy's argmax: the first NaN if any, else the first maximum.
__device__ __forceinline__ bool arg_better(float a, int ia, float b, int ib) {
    const bool na = isnan(a), nb = isnan(b);
    if (na != nb) return na;
    if (na) return ia < ib;
    return a > b || (a == b && ia < ib);
}
// The same order without branches (lane masks combined bitwise), for
// reductions across lanes.
__device__ __forceinline__ bool arg_better_select(float a, int ia, float b, int ib) {
    const bool na = a != a, nb = b != b, first = ia < ib;
    return (na & (!nb | first)) | (!na & !nb & ((a > b) | ((a == b) & first)));
}

// Per-row combination of the head's block partials (numpy argmax rule).
__global__ __launch_bounds__(256) void head_argmax_kernel(const float* __restrict__ val, const int32_t* __restrict__ idx,
                                                          int nblk, int64_t* __restrict__ out) {
    __shared__ float bv[256];
    __shared__ int bi[256];
    const int row = blockIdx.x, t = threadIdx.x;
    float v = 0.f;
    int i = 0x7fffffff;
    // eight independent loads per thread per round (2048 partials per round)
    for (int b0 = 0; b0 < nblk; b0 += 8 * 256) {
        float ov[8];
        int oi[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int b = b0 + 256 * u + t;
            ov[u] = b < nblk ? val[size_t(row) * nblk + b] : 0.f;
            oi[u] = b < nblk ? idx[size_t(row) * nblk + b] : 0x7fffffff;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (oi[u] != 0x7fffffff && (i == 0x7fffffff || arg_better(ov[u], oi[u], v, i))) { v = ov[u]; i = oi[u]; }
    }
    bv[t] = v;
    bi[t] = i;
    __syncthreads();
    for (int m = 128; m > 0; m >>= 1) {
        if (t < m) {
            const int o = t + m;
            if (bi[o] != 0x7fffffff && (bi[t] == 0x7fffffff || arg_better(bv[o], bi[o], bv[t], bi[t]))) {
                bv[t] = bv[o];
                bi[t] = bi[o];
            }
        }
        __syncthreads();
    }
    if (t == 0) out[row] = bi[0];
}

// ---------------------------------------------------------------------------
// Head projection of 33..64 rows with column-owning waves.
//
// Block = one row tile of the a.R rows, 128 columns.  Wave w owns two
// 16-column tiles over all 64 rows, so every code word is fetched and unpacked
// once per block:
//  - B: each lane loads its own packed code words straight into registers.
//    Lane i+16q of column tile ct takes, for k-step s (64 k), the words
//    j = 8s+2q and 8s+2q+1 (chunks of 8 codes) of its column; unpacked
//    (even codes, odd codes) they are the 16 operand bytes of that lane.
//  - A: the rows' activations of one 256-group per step are staged in LDS
//    through registers; 16-byte piece p of row r sits at slot p ^ (r & 15), so
//    the 16 rows read by one k-group of lanes hit distinct banks.  Lane i+16q
//    reads activation words 2j..2j+3 of row i, the same chunks j.
//
// Steps (one 256-group each) are unrolled, so the register rings have
// compile-time slots and every load wait is exact.  A moves global ->
// registers (loaded one step before its store) -> LDS (stored two steps before
// its dots, three stages) -> MFMA; codes are DB steps ahead.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256, 2) void head_rows_kernel(MfmaArgs a) {
    constexpr int GS = kHidden / kGroup, DB = 2;
    constexpr int KW = GS * 64;                               // activation words per row
    constexpr int NSTAGE = 3;                                 // A stages in LDS
    constexpr int NSC = NSTAGE;                               // scale stages (with their A words)
    __shared__ __attribute__((aligned(16))) uint32_t sA[NSTAGE][kMT * 64];
    __shared__ __attribute__((aligned(16))) float s_sa[NSC][kMT];
    __shared__ __attribute__((aligned(16))) float s_ss[NSC][kMT];
    __shared__ __attribute__((aligned(16))) float s_nb[NSC][kMT];   // -sa * kDotBias (exact)
    __shared__ float s_bv[4][kMT];                            // per-wave row best
    __shared__ int s_bi[4][kMT];

    const int nt = int(blockIdx.x), nrows = a.R;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, q = lane >> 4;
    const BankView bv = bank_view(true);                      // a dense N32 bank
    const int a_r = tid >> 2, a_part = tid & 3;

    // ---- B: code words of step st for this lane ----
    // (the last block may reach past N: its tiles repeat the last one, never stored)
    const int ntile = min((kNT * nt >> 5) + w, a.N / 32 - 1);
    uint32_t bw[DB][2][8];          // [slot][ct][2s + e]
    uint32_t bm[DB][2];             // meta word (sw | off << 16) per column tile
    auto load_b = [&](int st, int slot) {
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
            const int col = 32 * ntile + 16 * ct + li;
            const uint32_t* src = a.codes + bv.word(col, st, GS) + (2 * q) * bv.stride();
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                bw[slot][ct][2 * s] = src[(8 * s) * bv.stride()];
                bw[slot][ct][2 * s + 1] = src[(8 * s + 1) * bv.stride()];
            }
            bm[slot][ct] = a.meta[bv.meta(col, st, GS)];
        }
    };
#pragma unroll
    for (int st = 0; st < DB; ++st) load_b(st, st);

    // ---- A: activation words of group g, 64 bytes per lane (dead rows repeat the last live one) ----
    const uint32_t* a_src = a.act_words + size_t(min(a_r, nrows - 1)) * KW + 16 * a_part;
    // register k of the staging thread holds piece 4 a_part + (k + a_part) % 4
    // of its row: the 8 lanes of each LDS store phase (2 rows x 4 parts) then
    // hit 8 distinct 16-byte bank groups
    auto a_piece = [&](int k) { return (k + a_part) & 3; };
    const size_t sa_base = size_t(min(tid & 63, nrows - 1)) * GS;
    u32x4 ra[1][4];                 // one register slot: A(g) is loaded one step before its LDS store
    uint32_t rsa[1];
    int rsum[1];
    auto load_a = [&](int g, int slot) {
#pragma unroll
        for (int k = 0; k < 4; ++k) ra[slot][k] = *reinterpret_cast<const u32x4*>(a_src + g * 64 + 4 * a_piece(k));
        rsa[slot] = a.act_scales[sa_base + g];
        rsum[slot] = a.act_sums[sa_base + g];
    };
    auto store_a = [&](int slot, int stage, int g) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int piece = (4 * a_part + a_piece(k)) ^ (a_r & 15);
            *reinterpret_cast<u32x4*>(&sA[stage][a_r * 64 + 4 * piece]) = ra[slot][k];
        }
        if (tid < kMT) {
            const int sc = g % NSC;
            const float sa = f16_bits_to_f32(uint16_t(rsa[slot]));
            s_sa[sc][tid] = sa;
            s_ss[sc][tid] = sa * float(rsum[slot]);
            s_nb[sc][tid] = -sa * kDotBias;
        }
    };
    // A(0) and A(1) in flight together (A(1) through prologue-only registers)
    u32x4 ra1[4];
    uint32_t rsa1;
    int rsum1;
    load_a(0, 0);
#pragma unroll
    for (int k = 0; k < 4; ++k) ra1[k] = *reinterpret_cast<const u32x4*>(a_src + 64 + 4 * a_piece(k));
    rsa1 = a.act_scales[sa_base + 1];
    rsum1 = a.act_sums[sa_base + 1];
    store_a(0, 0, 0);
#pragma unroll
    for (int k = 0; k < 4; ++k) ra[0][k] = ra1[k];
    rsa[0] = rsa1;
    rsum[0] = rsum1;
    store_a(0, 1, 1);
    load_a(2, 0);
    __syncthreads();

    uint32_t flags = 0;
    // L = row tiles of 16 rows (dead rows repeat the last live one)
    auto run = [&]<int L>() {
        float val[4][2][4];
#pragma unroll
        for (int rt = 0; rt < 4; ++rt)
#pragma unroll
            for (int ct = 0; ct < 2; ++ct)
#pragma unroll
                for (int r = 0; r < 4; ++r) val[rt][ct][r] = 0.f;
        i32x4 acc[1][4][2];
        float swv[1][2], offv[1][2];
        constexpr i32x4 kAccInit = {kDotBiasBits, kDotBiasBits, kDotBiasBits, kDotBiasBits};

        // matrix-core dots of step ST for the L live row tiles (rows past
        // nrows in them hold copies of a live row)
        auto mfma_step = [&]<int ST>() {
            constexpr int stage = ST % NSTAGE, bslot = ST % DB, ab = 0;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                i32x4 fa[4], fb[2];
#pragma unroll
                for (int rt = 0; rt < L; ++rt) {
                    const int row = 16 * rt + li;
                    const u32x4 v = *reinterpret_cast<const u32x4*>(&sA[stage][row * 64 + 4 * ((4 * s + q) ^ li)]);
                    fa[rt] = i32x4{int(v.x), int(v.y), int(v.z), int(v.w)};
                }
#pragma unroll
                for (int ct = 0; ct < 2; ++ct) {
                    const uint32_t w0 = bw[bslot][ct][2 * s], w1 = bw[bslot][ct][2 * s + 1];
                    fb[ct] = i32x4{code_even(w0), code_odd(w0), code_even(w1), code_odd(w1)};
                }
#pragma unroll
                for (int rt = 0; rt < L; ++rt)
#pragma unroll
                    for (int ct = 0; ct < 2; ++ct)
                        acc[ab][rt][ct] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                            fa[rt], fb[ct], s ? acc[ab][rt][ct] : kAccInit, 0, 0, 0);
            }
            // the slot's scales are taken before the slot is refilled
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) {
                swv[ab][ct] = f16_bits_to_f32(uint16_t(bm[bslot][ct] & 0xffffu));
                offv[ab][ct] = f16_bits_to_f32(uint16_t(bm[bslot][ct] >> 16));
            }
            if constexpr (ST + DB < GS) load_b(ST + DB, bslot);
        };

        // fp32 group tree of step ST (dense_g256_api.h:35-37), ascending groups
        auto tree_step = [&]<int ST>() {
            constexpr int g = ST, sc = g % NSC, ab = 0;
#pragma unroll
            for (int rt = 0; rt < L; ++rt) {
                const float4 sa4 = *reinterpret_cast<const float4*>(&s_sa[sc][16 * rt + 4 * q]);
                const float4 ss4 = *reinterpret_cast<const float4*>(&s_ss[sc][16 * rt + 4 * q]);
                const float4 nb4 = *reinterpret_cast<const float4*>(&s_nb[sc][16 * rt + 4 * q]);
                const float sa[4] = {sa4.x, sa4.y, sa4.z, sa4.w}, ss[4] = {ss4.x, ss4.y, ss4.z, ss4.w};
                const float nb[4] = {nb4.x, nb4.y, nb4.z, nb4.w};
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int ct = 0; ct < 2; ++ct) {
                        // acc holds the bits of kDotBias + dot, one fma gives RN(sa * dot)
                        const float scaled_dot = __builtin_fmaf(sa[r], __int_as_float(acc[ab][rt][ct][r]), nb[r]);
                        const float product = swv[ab][ct] * scaled_dot;
                        const float correction = offv[ab][ct] * ss[r];
                        val[rt][ct][r] = val[rt][ct][r] + (product + correction);
                    }
            }
            // keep each step's tree in its step: sinking it would keep every
            // step's accumulators alive at once
#pragma unroll
            for (int rt = 0; rt < L; ++rt)
#pragma unroll
                for (int ct = 0; ct < 2; ++ct)
#pragma unroll
                    for (int r = 0; r < 4; ++r) asm volatile("" : "+v"(val[rt][ct][r]));
            if constexpr (g == GS - 1) {
                // ---- epilogue ----
                // Logits go through LDS (the A ring is free once every
                // wave is past its last dots) and leave as whole 16-byte
                // row pieces; per row, the best of this block's 128
                // columns (numpy argmax rule): lane (2 columns), 16 lanes
                // (xor 1..8), 4 waves in LDS.
                constexpr int kLS = kNT + 4;                  // padded row stride (floats)
                static_assert(kMT * kLS <= NSTAGE * kMT * 64, "logit staging fits the A ring");
                float* sL = reinterpret_cast<float*>(&sA[0][0]);
                const int nblk = (a.N + kNT - 1) / kNT;
                __syncthreads();
#pragma unroll
                for (int rt = 0; rt < L; ++rt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int row = 16 * rt + 4 * q + r;
                        float bv = 0.f;
                        int bi = 0x7fffffff;
#pragma unroll
                        for (int ct = 0; ct < 2; ++ct) {
                            const int cl = 32 * w + 16 * ct + li, col = kNT * nt + cl;
                            const float v = val[rt][ct][r];
                            sL[row * kLS + cl] = v;
                            if (col < a.N && (bi == 0x7fffffff || arg_better(v, col, bv, bi))) {
                                bv = v;
                                bi = col;
                            }
                            val[rt][ct][r] = 0.f;
                        }
#pragma unroll
                        for (int m = 1; m < 16; m <<= 1) {
                            float ov;
                            int oi;
                            if (m == 1) { ov = xor_perm_f<1>(bv); oi = xor_perm_i<1>(bi); }
                            else if (m == 2) { ov = xor_perm_f<2>(bv); oi = xor_perm_i<2>(bi); }
                            else if (m == 4) { ov = xor_perm_f<4>(bv); oi = xor_perm_i<4>(bi); }
                            else { ov = xor_perm_f<8>(bv); oi = xor_perm_i<8>(bi); }
                            if (oi != 0x7fffffff && (bi == 0x7fffffff || arg_better(ov, oi, bv, bi))) {
                                bv = ov;
                                bi = oi;
                            }
                        }
                        if (li == 0) { s_bv[w][row] = bv; s_bi[w][row] = bi; }
                    }
                __syncthreads();
                // rows of 32 float4 pieces: thread -> (row, piece), 8 rows per pass
                const int cols = min(kNT, a.N - kNT * nt);
                for (int row = tid >> 5; row < nrows; row += 8) {
                    const int c4 = 4 * (tid & 31);
                    if (c4 < cols) {
                        const float4 v = *reinterpret_cast<const float4*>(&sL[row * kLS + c4]);
                        const size_t o = size_t(row) * a.N + kNT * nt + c4;
                        *reinterpret_cast<float4*>(a.out + o) = v;
                        const float vv[4] = {v.x, v.y, v.z, v.w};
                        uint16_t b16[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            b16[e] = f32_to_bf16_bits(vv[e]);
                            if (!isfinite(vv[e])) flags |= a.flag_projection;
                            if ((b16[e] & 0x7f80u) == 0x7f80u) flags |= a.flag_bf16;
                        }
                        if (a.out_bf16)
                            *reinterpret_cast<uint2*>(a.out_bf16 + o) =
                                make_uint2(b16[0] | (uint32_t(b16[1]) << 16), b16[2] | (uint32_t(b16[3]) << 16));
                    }
                }
                if (tid < nrows) {
                    float bv = s_bv[0][tid];
                    int bi = s_bi[0][tid];
#pragma unroll
                    for (int ww = 1; ww < 4; ++ww) {
                        const float ov = s_bv[ww][tid];
                        const int oi = s_bi[ww][tid];
                        if (oi != 0x7fffffff && (bi == 0x7fffffff || arg_better(ov, oi, bv, bi))) {
                            bv = ov;
                            bi = oi;
                        }
                    }
                    a.arg_val[size_t(tid) * nblk + nt] = bv;
                    a.arg_idx[size_t(tid) * nblk + nt] = bi;
                }
            }
        };

        [&]<int... S>(std::integer_sequence<int, S...>) {
            ([&] {
                constexpr int ST = S;
                __syncthreads();            // A of step ST visible; stage (ST+2)%3 free
                if constexpr (ST + 2 < GS) {
                    store_a(0, (ST + 2) % NSTAGE, ST + 2);
                    if constexpr (ST + 3 < GS) load_a(ST + 3, 0);
                }
                mfma_step.template operator()<ST>();
                tree_step.template operator()<ST>();
            }(), ...);
        }(std::make_integer_sequence<int, GS>{});
    };
    run.template operator()<kMT / 16>();
    flag_or(a.sticky, flags);
}

// Every fp32 bit pattern (64 per thread): silu_portable_fast against
// silu_portable wherever silu_fast_domain holds.
__global__ __launch_bounds__(256) void silu_selfcheck_kernel(unsigned long long* checked, uint32_t* mismatches) {
    const uint64_t base = (uint64_t(blockIdx.x) * 256u + threadIdx.x) * 64u;
    unsigned long long n = 0;
    uint32_t bad = 0;
    for (int i = 0; i < 64; ++i) {
        const float g = __uint_as_float(uint32_t(base + i));
        if (!silu_fast_domain(g)) continue;
        ++n;
        bad += __float_as_uint(silu_portable(g)) != __float_as_uint(silu_portable_fast(g)) ? 1u : 0u;
    }
    atomicAdd(checked, n);
    if (bad) atomicAdd(mismatches, bad);
}

hipError_t launch_silu_selfcheck(unsigned long long* checked, uint32_t* mismatches, hipStream_t s) {
    // the counters are cleared by a kernel (graph-safe, no memset node)
    hipError_t st = launch_fill_u32(reinterpret_cast<uint32_t*>(checked), 2, 0u, s);
    if (st == hipSuccess) st = launch_fill_u32(mismatches, 1, 0u, s);
    if (st != hipSuccess) return st;
    timed_launch("silu_selfcheck", silu_selfcheck_kernel, dim3((1u << 26) / 256), dim3(256), 0, s, checked,
                 mismatches);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// G256 LM head for up to 32 rows on the 32x32x32 int8 matrix cores.
//
// A block of WPB waves copies the rows' A8 activations (32 rows x 2048 int8,
// rows past R repeating row R - 1) and per-group scales into LDS once; then
// every wave streams its own contiguous range of 32-column code tiles (the
// N / 32 tiles split evenly over the grid's waves) with D group-steps of
// codes in flight, the ring running across tiles.
//  - Codes of one (tile, group) are 32 rows j of 32 words (word (j, n): the 8
//    codes of column n for k = 8j .. 8j + 7).  Load u (0..15) of lane
//    n + 32h takes word (4 (u / 2) + 2h + u % 2, n): the 32 lanes of a half
//    read one whole 128-byte row, and lane n + 32h ends up holding column n,
//    rows 4i + 2h and 4i + 2h + 1 for MFMA i (0..7): its 16 operand bytes
//    (even codes, odd codes per word) of k-half h.
//  - A: lane r + 32h of MFMA i reads the matching activation words (chunks
//    4i + 2h, 4i + 2h + 1 of the group: 16-byte piece 2i + h); row r's piece
//    p sits at LDS slot (p & ~15) | ((p ^ r) & 15).
//  - Output register k of lane l is C[8 (k / 4) + 4 (l / 32) + k % 4][l % 32]:
//    the fp32 group tree (dense_g256_api.h:35-37) runs per lane over its 16
//    rows of one column, ascending groups.
// Logits leave straight from that layout (two 128-byte rows per store).  A
// lane meets its columns in ascending order, so its running argmax candidate
// per row changes only on a strictly larger value or a first NaN (numpy
// rule); the wave writes one partial per row at the end.
// ---------------------------------------------------------------------------
typedef int i32x16 __attribute__((ext_vector_type(16)));

template <int WPB, int D>
__global__ __launch_bounds__(64 * WPB, 1) void head_tile_kernel(MfmaArgs a, int nwaves) {
    constexpr int GS = kHidden / kGroup;          // 8 groups of 256
    constexpr int RW = kHidden / 4;               // activation words per row
    constexpr int ROWS = 32, NT = 64 * WPB;
    static_assert(GS % D == 0, "ring slots repeat every tile");
    __shared__ __attribute__((aligned(16))) uint32_t sA[ROWS * RW];
    __shared__ __attribute__((aligned(16))) float s_sa[GS][ROWS];
    __shared__ __attribute__((aligned(16))) float s_ss[GS][ROWS];
    __shared__ __attribute__((aligned(16))) float s_nb[GS][ROWS];   // -sa * kDotBias (exact)
    __shared__ uint64_t s_key[WPB][16][65];       // per-wave argmax keys (padded rows)
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int cl = lane & 31, h = lane >> 5;
    const int R = a.R;

    constexpr int APASS = ROWS * 128 / NT;        // 16-byte pieces per thread
    static_assert(APASS % 4 == 0, "pieces move in batches of four");
#pragma unroll
    for (int b = 0; b < APASS; b += 4) {
        u32x4 v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int i = (b + k) * NT + tid, r = i >> 7, pc = i & 127;
            v[k] = *reinterpret_cast<const u32x4*>(a.act_words + size_t(min(r, R - 1)) * RW + 4 * pc);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int i = (b + k) * NT + tid, r = i >> 7, pc = i & 127;
            *reinterpret_cast<u32x4*>(&sA[r * RW + 4 * ((pc & ~15) | ((pc ^ r) & 15))]) = v[k];
        }
    }
    for (int i = tid; i < ROWS * GS; i += NT) {
        const int r = i / GS, g = i % GS, sr = min(r, R - 1);
        const float sa = f16_bits_to_f32(a.act_scales[sr * GS + g]);
        s_sa[g][r] = sa;
        s_ss[g][r] = sa * float(a.act_sums[sr * GS + g]);
        s_nb[g][r] = -sa * kDotBias;
    }
    __syncthreads();

    // wave rank w * blocks + block: the ranks holding one tile more than the
    // rest (the lowest ones) spread over every CU, not a few whole blocks
    const int gw = w * int(gridDim.x) + int(blockIdx.x);
    if (gw >= nwaves) return;                     // no barrier follows
    const int ntiles = a.N >> 5;
    const int base = ntiles / nwaves, extra = ntiles % nwaves;
    const int c0 = gw * base + min(gw, extra), cnt = base + (gw < extra ? 1 : 0);

    // step st = 8 * (tile - c0) + group: 1024 code words and 32 meta words on
    const uint32_t* cbase = a.codes + size_t(c0) * GS * 1024 + 64 * h + cl;
    const uint32_t* mbase = a.meta + size_t(c0) * GS * 32 + cl;
    uint32_t bw[D][16];
    uint32_t bm[D];
    auto load_b = [&](int st, int slot) {
        const uint32_t* src = cbase + size_t(st) * 1024;
#pragma unroll
        for (int u = 0; u < 16; ++u) bw[slot][u] = load_once(src + 128 * (u >> 1) + 32 * (u & 1));
        bm[slot] = mbase[size_t(st) * 32];
    };
#pragma unroll
    for (int st = 0; st < D; ++st) load_b(st, st);

    // candidate per row: value and tile (t < 256: one byte each, packed);
    // all -inf keeps the first tile (the first column)
    float bv[16];
    uint32_t bt[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int k = 0; k < 16; ++k) bv[k] = -__builtin_inff();
    float nonfinite = 0.f, nonfinite_bf16 = 0.f;  // NaN once a logit (resp. its bf16) is inf or NaN
    constexpr i32x16 kAccInit = {kDotBiasBits, kDotBiasBits, kDotBiasBits, kDotBiasBits, kDotBiasBits, kDotBiasBits,
                                 kDotBiasBits, kDotBiasBits, kDotBiasBits, kDotBiasBits, kDotBiasBits, kDotBiasBits,
                                 kDotBiasBits, kDotBiasBits, kDotBiasBits, kDotBiasBits};

    // one code tile: 8 groups; REFILL = a next tile exists
    auto tile_body = [&]<bool REFILL>(int t) {
        float val[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) val[k] = 0.f;
#pragma unroll
        for (int g = 0; g < GS; ++g) {
            const int slot = g % D;
            i32x16 acc;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t w0 = bw[slot][2 * i], w1 = bw[slot][2 * i + 1];
                const i32x4 fb = {code_even(w0), code_odd(w0), code_even(w1), code_odd(w1)};
                const u32x4 av =
                    *reinterpret_cast<const u32x4*>(&sA[cl * RW + 4 * ((16 * g) | ((2 * i + h) ^ (cl & 15)))]);
                const i32x4 fa = {int(av.x), int(av.y), int(av.z), int(av.w)};
                acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa, fb, i ? acc : kAccInit, 0, 0, 0);
            }
            // pin the meta word here: left free, its conversion is hoisted
            // next to the load and waits out the whole ring
            asm volatile("" : "+v"(bm[slot]));
            const float sw = f16_bits_to_f32(uint16_t(bm[slot] & 0xffffu));
            const float off = f16_bits_to_f32(uint16_t(bm[slot] >> 16));
            if (g + D < GS) load_b(8 * t + g + D, slot);
            else if constexpr (REFILL) load_b(8 * t + g + D, slot);
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const float4 sa4 = *reinterpret_cast<const float4*>(&s_sa[g][8 * b + 4 * h]);
                const float4 ss4 = *reinterpret_cast<const float4*>(&s_ss[g][8 * b + 4 * h]);
                const float4 nb4 = *reinterpret_cast<const float4*>(&s_nb[g][8 * b + 4 * h]);
                const float sa[4] = {sa4.x, sa4.y, sa4.z, sa4.w}, ss[4] = {ss4.x, ss4.y, ss4.z, ss4.w};
                const float nb[4] = {nb4.x, nb4.y, nb4.z, nb4.w};
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int k = 4 * b + c;
                    const float scaled_dot = __builtin_fmaf(sa[c], __int_as_float(acc[k]), nb[c]);
                    const float product = sw * scaled_dot;
                    const float correction = off * ss[c];
                    val[k] = val[k] + (product + correction);
                }
            }
#pragma unroll
            for (int k = 0; k < 16; ++k) asm volatile("" : "+v"(val[k]));
        }
        // rows past R repeat row R - 1 bit for bit, so every lane's values
        // may feed the flags and the candidates
        const int col = 32 * (c0 + t) + cl;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const int row = 8 * (k >> 2) + 4 * h + (k & 3);
            const float v = val[k];
            const uint16_t b16 = f32_to_bf16_bits(v);
            if (row < R) {
                const size_t o = size_t(row) * a.N + col;
                a.out[o] = v;
                if (a.out_bf16) a.out_bf16[o] = b16;
            }
            nonfinite = __builtin_fmaf(v, 0.f, nonfinite);
            nonfinite_bf16 = __builtin_fmaf(bf16_bits_to_f32(b16), 0.f, nonfinite_bf16);
            const bool take = (v > bv[k]) | ((v != v) & (bv[k] == bv[k]));
            bv[k] = take ? v : bv[k];
            const uint32_t mask = 0xffu << (8 * (k & 3));
            bt[k >> 2] = take ? ((bt[k >> 2] & ~mask) | (uint32_t(t) << (8 * (k & 3)))) : bt[k >> 2];
        }
    };
    for (int t = 0; t + 1 < cnt; ++t) tile_body.template operator()<true>(t);
    tile_body.template operator()<false>(cnt - 1);

    // ---- per-row best of the wave, then one partial per row.  Key: an
    // order-preserving image of the value (-0 as +0, every NaN above +inf)
    // over the complemented column, so the unsigned maximum is the numpy
    // argmax candidate (first NaN, else first maximum).  The 16 keys of each
    // lane go through LDS; lane r (and r + 32) takes row r's 32 candidates
    // (columns cl of its half), 16 each, and the two halves meet by xor 32.
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const float v = bv[k] + 0.f;
        const uint32_t u = __float_as_uint(v);
        const uint32_t ord = v != v ? 0xffffffffu : ((u & 0x80000000u) ? ~u : (u | 0x80000000u));
        const int colk = 32 * (c0 + int((bt[k >> 2] >> (8 * (k & 3))) & 0xffu)) + cl;
        s_key[w][k][lane] = (uint64_t(ord) << 32) | uint32_t(~colk);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    {
        const int r = lane & 31, rh = (r >> 2) & 1, rk = 4 * (r >> 3) + (r & 3), c0h = 16 * (lane >> 5);
        uint64_t key = s_key[w][rk][32 * rh + c0h];
#pragma unroll
        for (int c = 1; c < 16; ++c) {
            const uint64_t o = s_key[w][rk][32 * rh + c0h + c];
            key = o > key ? o : key;
        }
        const int hi = xor_perm_i<32>(int(key >> 32)), lo = xor_perm_i<32>(int(uint32_t(key)));
        const uint64_t other = (uint64_t(uint32_t(hi)) << 32) | uint32_t(lo);
        key = other > key ? other : key;
        if (lane < 32 && r < R) {
            const uint32_t o = uint32_t(key >> 32);
            const float v = o == 0xffffffffu ? __builtin_nanf("") : __uint_as_float((o & 0x80000000u) ? (o & 0x7fffffffu) : ~o);
            a.arg_idx[size_t(r) * nwaves + gw] = int(~uint32_t(key));
            a.arg_val[size_t(r) * nwaves + gw] = v;
        }
    }
    uint32_t flags = 0;
    if (nonfinite != nonfinite) flags |= a.flag_projection;
    if (nonfinite_bf16 != nonfinite_bf16) flags |= a.flag_bf16;
    flag_or(a.sticky, flags);
}

// Head waves: WPB-wave blocks (one per CU), at least two code tiles per wave
// (so the partial count per row, nwaves, stays within ceil(N / 64)).
constexpr int kHeadWaves = 8, kHeadRing = 2;
static int head_waves(int N) { return std::max(1, std::min(kHeadWaves * device_cu_count(), (N / 32) / 2)); }

hipError_t launch_head_mfma(const MfmaArgs& a, int64_t* argmax, hipStream_t s) {
    if (a.R <= 0 || a.R > kMT || a.N <= 0 || a.N % 32 != 0 || a.K != kHidden) return hipErrorInvalidValue;
    int nparts;
    if (a.R <= 32) {
        // up to 32 rows (the decode-side head): streaming waves
        nparts = head_waves(a.N);
        timed_launch("head_mfma", head_tile_kernel<kHeadWaves, kHeadRing>,
                     dim3((nparts + kHeadWaves - 1) / kHeadWaves), dim3(64 * kHeadWaves), 0, s, a, nparts);
    } else {
        nparts = (a.N + kNT - 1) / kNT;
        timed_launch("head_mfma", head_rows_kernel, dim3(nparts), dim3(256), 0,
                     s, a);
    }
    hipError_t st = hipGetLastError();
    if (st != hipSuccess) return st;
    timed_launch("argmax", head_argmax_kernel, dim3(a.R), dim3(256), 0, s, a.arg_val, a.arg_idx, nparts, argmax);
    return hipGetLastError();
}

}  // namespace ornith
