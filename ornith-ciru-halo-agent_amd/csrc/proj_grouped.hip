// Grouped G256 projections of the permuted routes on the int8 matrix cores
// (layers of more than 32 tokens).
//
// Arithmetic is the reference's A8/A4 routed math, exactly
// (routed_storage_n32_prefill.h:43-149 computes the same per-group integer
// dots with WMMA-iu4, routed_storage_n32_consumer.cpp:152-157 the tree):
// per (route, column, 256-group) the integer dot sum_k code*q is formed by
// v_mfma_i32_16x16x64_i8 (exact: |dot| < 2^19), then the fp32 group tree
// value = value + (RN(sw*RN(sa*dot)) + RN(off*RN(sa*sum))) runs in ascending
// group order.
//
// MFMA operand layout (verified on gfx950): lane i+16q supplies the 16 bytes
// of row/column i for k-group q, A and B bytes pair positionally, and output
// register r of lane l is C[4*(l/16)+r][l%16].
//
// Which 16 columns share a product is free, so the columns are dealt for the
// loads: a wave owns two 32-column tiles, lane li = l % 16 takes the four
// consecutive columns 4 (li % 8) .. + 3 of tile li / 8, and product ct is made
// of every lane's ct-th one.  One 16-byte load then carries the same eight
// k values of four columns (two whole 128-byte rows of an N32 tile per 16
// lanes), and a lane ends with four consecutive columns of a row: one 16-byte
// store.
#include "kernels.hpp"
#include "timing.hpp"
#include "decode.hpp"
#include "mfma.hpp"

namespace ornith {
namespace {


// ---- pieces shared by both projections -----------------------------------------
// Code words of one 256-group of a wave's 64 columns: raw[s][e][ct] is the
// word of chunk 8 s + 4 e + q (8 codes) of the lane's column ct; the 16 B
// bytes of k-step s are (even codes, odd codes) of e = 0, 1.  (The four
// k-groups of lanes take consecutive chunks, so a load covers whole cache
// lines of an N16 tile too.)
struct Codes {
    u32x4 raw[4][2];
    u32x4 meta;                      // scale | offset << 16 of the four columns
};
// metadata pointers are only known to be 4-byte aligned
typedef u32x4 u32x4_a4 __attribute__((aligned(4)));
__device__ __forceinline__ i32x4 b_operand(const Codes& c, int s, int ct) {
    const uint32_t w0 = c.raw[s][0][ct], w1 = c.raw[s][1][ct];
    return i32x4{code_even(w0), code_odd(w0), code_even(w1), code_odd(w1)};
}

template <bool ONCE> __device__ __forceinline__ u32x4 load16(const char* p) {
    if constexpr (ONCE) return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
    else return *reinterpret_cast<const u32x4*>(p);
}

// The bank of a block (tiles of TW columns) and the lane's place in it: byte
// offset of chunk q of the lane's first column (group 0) and of its
// metadata.
template <int TW> struct BankLane {
    static constexpr int kChunk = TW * 4, kGroupBytes = 32 * kChunk;   // bytes from a chunk / a group to the next
    const char* codes;
    const char* meta;
    uint32_t word, mword;
    __device__ __forceinline__ BankLane(const uint32_t* c, const uint32_t* m, int col, int groups, int q)
        : codes(reinterpret_cast<const char*>(c)), meta(reinterpret_cast<const char*>(m)) {
        constexpr BankView bv{TW == 16 ? 4 : 5};
        word = uint32_t(bv.word(col, 0, groups) + q * TW) * 4u;
        mword = uint32_t(bv.meta(col, 0, groups)) * 4u;
    }
    // the words of k-step s of group g
    template <bool ONCE> __device__ __forceinline__ void load(Codes& c, int s, int g) const {
        const char* src = codes + size_t(g) * kGroupBytes;
#pragma unroll
        for (int e = 0; e < 2; ++e) c.raw[s][e] = load16<ONCE>(src + (8 * s + 4 * e) * kChunk + word);
    }
    __device__ __forceinline__ void load_meta(Codes& c, int g) const {
        c.meta = *reinterpret_cast<const u32x4_a4*>(meta + size_t(g) * kChunk + mword);
    }
    template <bool ONCE> __device__ __forceinline__ void load_all(Codes& c, int g) const {
#pragma unroll
        for (int s = 0; s < 4; ++s) load<ONCE>(c, s, g);
        load_meta(c, g);
    }
    // the same lane `cols` columns on (a multiple of 32), K = 256 groups
    __device__ __forceinline__ BankLane ahead(int cols, int groups) const {
        BankLane b = *this;
        b.codes += size_t(cols) * groups * (kGroup / 2);
        b.meta += size_t(cols) * groups * 4;
        return b;
    }
};

// Activations of MT rows x GS groups in LDS: 16-byte piece 4 s + q of row r in
// group g holds chunks 8 s + q and 8 s + 4 + q (what lane q multiplies in
// k-step s), at slot (4 s + q) ^ (r & 15), so the 16 rows that a k-group of
// lanes reads hit distinct banks; scales, RN(scale * sum) and -scale * kDotBias
// beside them.
template <int MT, int GS> struct Rows {
    uint32_t words[GS][MT * 64];
    float sa[GS][MT], ss[GS][MT], nb[GS][MT];
    int src[MT];                     // activation row of each tile row (dead rows repeat the last live one)
    int route[MT];                   // its route, -1 for a dead row
};

// Copies the rows into LDS: the block's threads take consecutive pieces.
template <int MT, int GS, int THREADS>
__device__ __forceinline__ void stage_rows(Rows<MT, GS>& R, const MfmaArgs& a) {
    const int tid = threadIdx.x;
    constexpr int kPieces = MT * GS * 16 / THREADS;          // 16-byte pieces per thread
    constexpr int kBatch = kPieces < 8 ? kPieces : 8;
#pragma unroll
    for (int b = 0; b < kPieces; b += kBatch) {
        u32x4 v[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
            const int i = (b + k) * THREADS + tid, row = i / (GS * 16), pc = i % (GS * 16);
            v[k] = *reinterpret_cast<const u32x4*>(a.act_words + size_t(R.src[row]) * (GS * 64) + 4 * pc);
        }
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
            const int i = (b + k) * THREADS + tid, row = i / (GS * 16), pc = i % (GS * 16);
            // chunks 2 p and 2 p + 1 of the group (p = pc % 16): half (p % 4) / 2 of pieces 4 s + 2 (p % 2) + 0, 1
            const int p = pc & 15, to = (p & 12) | (2 * (p & 1)), half = p & 2;
            uint32_t* dst = &R.words[pc >> 4][row * 64 + half];
            *reinterpret_cast<uint2*>(dst + 4 * (to ^ (row & 15))) = make_uint2(v[k].x, v[k].y);
            *reinterpret_cast<uint2*>(dst + 4 * ((to + 1) ^ (row & 15))) = make_uint2(v[k].z, v[k].w);
        }
    }
    for (int i = tid; i < MT * GS; i += THREADS) {
        const int row = i / GS, g = i % GS;
        const size_t at = size_t(R.src[row]) * GS + g;
        const float sa = f16_bits_to_f32(a.act_scales[at]);
        R.sa[g][row] = sa;
        R.ss[g][row] = sa * float(a.act_sums[at]);
        R.nb[g][row] = -sa * kDotBias;
    }
}

// Dots and fp32 tree of one 256-group for L row tiles of 16 rows.
// val[rt][ct][r]: row 16 rt + 4 q + r, column ct of the lane.  Each k-step's
// words are refilled with group gnext of `next` as soon as they are unpacked,
// so a wave always has about 8 KiB of codes in flight (REFILL false: the
// wave's last step, nothing is left to load).
template <int L, bool ONCE, bool REFILL = true, int MT, int GS, int TW>
__device__ __forceinline__ void group_step(const Rows<MT, GS>& R, Codes& c, int g, float (&val)[L][4][4],
                                           const BankLane<TW>& next, int gnext) {
    const int lane = threadIdx.x & 63, li = lane & 15, q = lane >> 4;
    constexpr i32x4 kInit = {kDotBiasBits, kDotBiasBits, kDotBiasBits, kDotBiasBits};
    float sw[4];
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) sw[ct] = f16_bits_to_f32(c.meta[ct] & 0xffffu);
    const uint32_t om = q < 2 ? (q == 0 ? c.meta[0] : c.meta[1]) : (q == 2 ? c.meta[2] : c.meta[3]);
    const float off = f16_bits_to_f32(om >> 16);
    i32x4 acc[L][4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        i32x4 fb[4];
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) fb[ct] = b_operand(c, s, ct);
        if constexpr (REFILL) next.template load<ONCE>(c, s, gnext);
#pragma unroll
        for (int rt = 0; rt < L; ++rt) {
            const u32x4 v =
                *reinterpret_cast<const u32x4*>(&R.words[g][(16 * rt + li) * 64 + 4 * ((4 * s + q) ^ li)]);
            const i32x4 fa = {int(v.x), int(v.y), int(v.z), int(v.w)};
#pragma unroll
            for (int ct = 0; ct < 4; ++ct)
                acc[rt][ct] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa, fb[ct], s ? acc[rt][ct] : kInit, 0, 0, 0);
        }
    }
    if constexpr (REFILL) next.load_meta(c, gnext);
#pragma unroll
    for (int rt = 0; rt < L; ++rt) {
        // RN(offset * RN(sa * sum)) of the lane's four columns x four rows by
        // one exact K = 1 product instead of 16 multiplications: its block
        // b = lane / 16 is column ct = b, so lane (li, q) supplies column q's
        // offset and row li's RN(sa * sum)
        const f32x16 zero = {};
        const f32x16 corr = __builtin_amdgcn_mfma_f32_16x16x1f32(R.ss[g][16 * rt + li], off, zero, 0, 0, 0);
        const f32x4 sa = *reinterpret_cast<const f32x4*>(&R.sa[g][16 * rt + 4 * q]);
        const f32x4 nb = *reinterpret_cast<const f32x4*>(&R.nb[g][16 * rt + 4 * q]);
#pragma unroll
        for (int ct = 0; ct < 4; ++ct)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float scaled_dot = __builtin_fmaf(sa[r], __int_as_float(acc[rt][ct][r]), nb[r]);
                const float product = sw[ct] * scaled_dot;
                val[rt][ct][r] = val[rt][ct][r] + (product + corr[4 * ct + r]);
            }
    }
}

// Block -> (m-tile, column block nt of NCB).  Workgroups go to the 8 XCDs
// round-robin (linear block b runs on XCD b % 8): XCD x takes the contiguous
// m-tiles [x per, (x + 1) per), all column blocks of a tile in a row, so a
// tile's activation rows and the weights of an expert's consecutive m-tiles
// meet in one L2.  Against dealing column blocks first: gate-up 29.0 -> 24.0
// us at 256 tokens, 66.8 -> 61.8 at 1120, 296 -> 288 at 8192 (Zipf routing).
template <int NCB> __device__ __forceinline__ bool block_tile(const MfmaArgs& a, int& mtile, int& nt) {
    const int b = int(blockIdx.x), ntiles = a.ntiles[0], per = (ntiles + 7) >> 3, k = b / (8 * NCB);
    nt = (b >> 3) % NCB;
    mtile = (b & 7) * per + k;
    return k < per && mtile < ntiles;
}

// ---------------------------------------------------------------------------
// Gate-up: block (m-tile, half h): middle columns 256 h .. + 255, one whole
// 256-group of the down input.  Wave w's two tiles are gate and up of columns
// 256 h + 32 w .. + 31.  The block's SiLU(gate) * up rows meet in LDS, where
// H128 + quantisation turns them into the down projection's int8 words.
// ---------------------------------------------------------------------------
template <int MT, int WAVES, int QMAX, bool ONCE>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(MT == 16 ? 4 : 2, MT == 16 ? 4 : 2))) void
gateup_tile_kernel(MfmaArgs a) {
    constexpr int GS = kHidden / kGroup, PASSES = 8 / WAVES, kRow = kGroup + 4;    // padded middle row (floats)
    __shared__ __attribute__((aligned(16))) Rows<MT, GS> R;
    static_assert(sizeof(R.words) >= sizeof(float) * MT * kRow, "the middle rows reuse the activation words");
    int mtile, h;
    if (!block_tile<2>(a, mtile, h)) return;
    const Segment td = a.tiles[mtile];
    const int bank = td.bank, first = td.first, nrows = td.count;
    const bool shared = bank == kShared;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, q = lane >> 4, th = li >> 3;
    // (clamped to the route range: a malformed list gives wrong rows, never
    // an access outside the activation / output buffers)
    const int rmax = a.R + (a.shared_codes ? a.R / kTop : 0) - 1;
    const int route = min(max(a.routes[first + min(tid & (MT - 1), nrows - 1)], 0), rmax);
    __builtin_amdgcn_sched_barrier(0);
    uint32_t flags = 0;
    float* mid_rows = reinterpret_cast<float*>(&R.words[0][0]);
    auto body = [&]<int TW>(const uint32_t* codes, const uint32_t* meta) {
        const BankLane<TW> bank_at(codes, meta, (th ? kInter : 0) + kGroup * h + 32 * w + 4 * (li & 7), GS, q);
        Codes c;
        bank_at.template load_all<ONCE>(c, 0);
        if (tid < MT) R.src[tid] = route < a.R ? route / kTop : route - a.R;
        __syncthreads();
        stage_rows<MT, GS, 64 * WAVES>(R, a);
        __syncthreads();
        auto run = [&]<int L>() {
            float mid[PASSES][L][2][4];
            bool finite = true;
#pragma unroll
            for (int p = 0; p < PASSES; ++p) {
                const BankLane<TW> here = bank_at.ahead(32 * WAVES * p, GS);
                const BankLane<TW> after = bank_at.ahead(32 * WAVES * min(p + 1, PASSES - 1), GS);
                float val[L][4][4];
#pragma unroll
                for (int rt = 0; rt < L; ++rt)
#pragma unroll
                    for (int ct = 0; ct < 4; ++ct)
#pragma unroll
                        for (int r = 0; r < 4; ++r) val[rt][ct][r] = 0.f;
#pragma unroll 1
                for (int g = 0; g < GS - 1; ++g) group_step<L, ONCE>(R, c, g, val, here, g + 1);
                group_step<L, ONCE>(R, c, GS - 1, val, after, 0);
                // lanes li and li ^ 8 hold gate and up of the same columns: the gate
                // lane finishes rows 4q + 0, 1 of each row tile, the up lane 4q + 2, 3
#pragma unroll
                for (int rt = 0; rt < L; ++rt) {
                    float gate[2][4], up[2][4];
#pragma unroll
                    for (int k = 0; k < 2; ++k)
#pragma unroll
                        for (int ct = 0; ct < 4; ++ct) {
                            const float own = th ? val[rt][ct][2 + k] : val[rt][ct][k];
                            const float other = xor_perm_f<8>(th ? val[rt][ct][k] : val[rt][ct][2 + k]);
                            gate[k][ct] = th ? other : own;
                            up[k][ct] = th ? own : other;
                        }
                    if (shared) {
                        // shared linear outputs are bf16; tabulated SiLU; bf16 product
                        // (routed_storage_n32_consumer.cpp:226-227, 246-250)
#pragma unroll
                        for (int k = 0; k < 2; ++k)
#pragma unroll
                            for (int ct = 0; ct < 4; ++ct) {
                                gate[k][ct] = bf16_round(gate[k][ct]);
                                up[k][ct] = bf16_round(up[k][ct]);
                                mid[p][rt][k][ct] = bf16_round(a.silu_table[__float_as_uint(gate[k][ct]) >> 16] * up[k][ct]);
                                finite = finite && isfinite(gate[k][ct]) && isfinite(up[k][ct]);
                            }
                    } else {
                        // the short form when every gate value of the wave is in its
                        // domain (common.hpp), the full one otherwise
                        bool fast = true;
#pragma unroll
                        for (int k = 0; k < 2; ++k)
#pragma unroll
                            for (int ct = 0; ct < 4; ++ct) fast = fast && silu_fast_domain(gate[k][ct]);
                        if (__builtin_amdgcn_ballot_w64(!fast) == 0) {
#pragma unroll
                            for (int k = 0; k < 2; ++k)
#pragma unroll
                                for (int ct = 0; ct < 4; ++ct) mid[p][rt][k][ct] = silu_portable_fast(gate[k][ct]) * up[k][ct];
                        } else {
#pragma unroll
                            for (int k = 0; k < 2; ++k)
#pragma unroll
                                for (int ct = 0; ct < 4; ++ct) mid[p][rt][k][ct] = silu_portable(gate[k][ct]) * up[k][ct];
                        }
                    }
                    // a non-finite gate or up value of a routed expert always gives a
                    // non-finite middle value (NaN, inf * x, x / inf or 0 * inf; in the
                    // fast domain silu(g) is finite and nonzero).  Dead rows repeat a
                    // live row, flags included.
#pragma unroll
                    for (int k = 0; k < 2; ++k)
#pragma unroll
                        for (int ct = 0; ct < 4; ++ct) finite = finite && isfinite(mid[p][rt][k][ct]);
                    if (__builtin_amdgcn_ballot_w64(!finite) != 0) {
#pragma unroll
                        for (int k = 0; k < 2; ++k)
#pragma unroll
                            for (int ct = 0; ct < 4; ++ct) {
                                if (!isfinite(gate[k][ct]) || !isfinite(up[k][ct])) flags |= kFlagNonfiniteProjection;
                                if (!isfinite(mid[p][rt][k][ct])) flags |= kFlagNonfiniteMiddle | kFlagNonfiniteInput;
                            }
                    }
                }
            }
            __syncthreads();                                       // every wave is past its last dots
#pragma unroll
            for (int p = 0; p < PASSES; ++p)
#pragma unroll
                for (int rt = 0; rt < L; ++rt)
#pragma unroll
                    for (int k = 0; k < 2; ++k)
                        *reinterpret_cast<f32x4*>(mid_rows + (16 * rt + 4 * q + 2 * th + k) * kRow +
                                                  32 * (w + WAVES * p) + 4 * (li & 7)) =
                            f32x4{mid[p][rt][k][0], mid[p][rt][k][1], mid[p][rt][k][2], mid[p][rt][k][3]};
        };
        if (MT > 16 && nrows > 16) run.template operator()<MT / 16>();
        else run.template operator()<1>();
    };
    if (shared) body.template operator()<32>(a.shared_codes, a.shared_meta);
    else body.template operator()<kRoutedTile>(a.codes + size_t(bank) * a.bank_words,
                                               a.meta + size_t(bank) * a.bank_meta_words);
    __syncthreads();
    // H128 + quantisation, a quarter-wave per row (its group h)
    const int l = lane & 15;
    for (int r0 = 4 * w; r0 < nrows; r0 += 4 * WAVES) {       // wave-uniform
        const int row = r0 + (lane >> 4);
        const float* src = mid_rows + min(row, nrows - 1) * kRow + quarter_base(l);
        float v[16];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const f32x4 m = *reinterpret_cast<const f32x4*>(src + 4 * i);
            v[4 * i] = m[0]; v[4 * i + 1] = m[1]; v[4 * i + 2] = m[2]; v[4 * i + 3] = m[3];
        }
        h128_quarter(v);
        uint32_t w4[4], f = 0;
        uint16_t sbits;
        int sum;
        quantize_quarter_fast<QMAX>(v, w4, sbits, sum, f, kFlagNonfiniteInput | kFlagInvalidActivation,
                                    kFlagInvalidActivation);
        if (row < nrows) {
            const size_t at = size_t(first + row) * (kInter / kGroup) + h;
            *reinterpret_cast<uint4*>(a.mid_words + at * 64 + quarter_base(l) / 4) =
                make_uint4(w4[0], w4[1], w4[2], w4[3]);
            if (l == 0) { a.mid_scales[at] = sbits; a.mid_sums[at] = sum; }
            flags |= f;
        }
    }
    flag_or(a.sticky, flags);
}

// ---------------------------------------------------------------------------
// Down: block (m-tile, CH x 256 columns); wave w's chunk c is columns
// 256 (CH nt + c) + 64 w .. + 63.  Both groups (K = 512) of the rows are in LDS.
// Bound by the code stream at few tokens and by the fp32 route rows it writes
// at many (604 MB at 8192 tokens with the shared expert), so it wants waves in
// flight: 16-row blocks stay within 128 registers without scratch (four waves
// per SIMD), 32-row ones within 168 (three), which one loop over the group
// steps allows (unrolled by group it needs 230 and spills at 16 rows).  The
// wave's last step is outside the loop: it has no codes left to load.  With two
// waves per SIMD, 24 bytes of scratch at 16 rows and that refill of codes
// nobody used: 36.7 -> 32.2 us at 131 tokens, 68.3 -> 60.7 at 2048.
// ---------------------------------------------------------------------------
template <int MT, int WAVES, int CH, bool ONCE>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(MT == 16 ? 4 : 3, MT == 16 ? 4 : 3))) void
down_tile_kernel(MfmaArgs a) {
    constexpr int GS = kInter / kGroup, kCols = 64 * WAVES, NCB = kHidden / (kCols * CH);
    __shared__ __attribute__((aligned(16))) Rows<MT, GS> R;
    int mtile, nt;
    if (!block_tile<NCB>(a, mtile, nt)) return;
    const Segment td = a.tiles[mtile];
    const int bank = td.bank, first = td.first, nrows = td.count;
    const bool shared = bank == kShared;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, li = lane & 15, q = lane >> 4, th = li >> 3;
    const int rmax = a.R + (a.shared_codes ? a.R / kTop : 0) - 1;
    const int route = min(max(a.routes[first + min(tid & (MT - 1), nrows - 1)], 0), rmax);
    __builtin_amdgcn_sched_barrier(0);
    const int col0 = kCols * CH * nt + 64 * w + 32 * th + 4 * (li & 7);
    float nonfinite = 0.f;                                      // NaN once a value is inf or NaN
    auto body = [&]<int TW>(const uint32_t* codes, const uint32_t* meta) {
        const BankLane<TW> bank_at(codes, meta, col0, GS, q);
        Codes c;
        bank_at.template load_all<ONCE>(c, 0);
        if (tid < MT) {
            R.src[tid] = first + min(tid, nrows - 1);
            R.route[tid] = tid < nrows ? route : -1;
        }
        __syncthreads();
        stage_rows<MT, GS, 64 * WAVES>(R, a);
        __syncthreads();
        auto run = [&]<int L>() {
            float val[L][4][4];
#pragma unroll
            for (int rt = 0; rt < L; ++rt)
#pragma unroll
                for (int ct = 0; ct < 4; ++ct)
#pragma unroll
                    for (int r = 0; r < 4; ++r) val[rt][ct][r] = 0.f;
            auto finish = [&](int ch) {
#pragma unroll
                for (int rt = 0; rt < L; ++rt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        f32x4 v;
#pragma unroll
                        for (int ct = 0; ct < 4; ++ct) {
                            v[ct] = shared ? bf16_round(val[rt][ct][r]) : val[rt][ct][r];
                            nonfinite = __builtin_fmaf(v[ct], 0.f, nonfinite);
                            val[rt][ct][r] = 0.f;
                        }
                        const int to = R.route[16 * rt + 4 * q + r];
                        if (to >= 0) *reinterpret_cast<f32x4*>(a.out + size_t(to) * kHidden + col0 + kCols * ch) = v;
                    }
            };
            // step st: group st % 2 of chunk st / 2 (GS = 2), refilled with the next step's codes
#pragma unroll 1
            for (int st = 0; st < 2 * CH - 1; ++st) {
                group_step<L, ONCE>(R, c, st & 1, val, bank_at.ahead(kCols * ((st + 1) >> 1), GS), (st + 1) & 1);
                if (st & 1) finish(st >> 1);
            }
            group_step<L, ONCE, false>(R, c, 1, val, bank_at, 0);
            finish(CH - 1);
        };
        if (MT > 16 && nrows > 16) run.template operator()<MT / 16>();
        else run.template operator()<1>();
    };
    if (shared) body.template operator()<32>(a.shared_codes, a.shared_meta);
    else body.template operator()<kRoutedTile>(a.codes + size_t(bank) * a.bank_words,
                                               a.meta + size_t(bank) * a.bank_meta_words);
    flag_or(a.sticky, nonfinite != nonfinite ? kFlagNonfiniteProjection : 0u);
}

template <int MT, int GW, int DW, int CH, bool ONCE>
hipError_t launch_tiles(const MfmaArgs& a, bool gateup, int qmax, int max_tiles, hipStream_t s) {
    const int tiles8 = (max_tiles + 7) / 8 * 8;   // m-tiles rounded up to the 8 XCDs
    if (gateup && qmax == 127)
        timed_launch("gateup_mfma", gateup_tile_kernel<MT, GW, 127, ONCE>, dim3(tiles8 * 2), dim3(64 * GW), 0, s, a);
    else if (gateup)
        timed_launch("gateup_mfma", gateup_tile_kernel<MT, GW, 7, ONCE>, dim3(tiles8 * 2), dim3(64 * GW), 0, s, a);
    else
        timed_launch("down_mfma", down_tile_kernel<MT, DW, CH, ONCE>, dim3(tiles8 * (kHidden / (64 * DW * CH))),
                     dim3(64 * DW), 0, s, a);
    return hipGetLastError();
}

}  // namespace

// Rows per m-tile.  Few routes per expert: 16-row tiles, whose kernels keep
// four waves per SIMD streaming codes; with more routes 32-row tiles read the
// codes and unpack them half as often.  Between 200 and 1100 tokens the better
// height follows the number of 32-row gate-up blocks against the chip's 512
// slots, which hangs on the routing: spread evenly over the experts it ends up
// just past a round of them, skewed well below.  T is all the host knows, so
// each line lies where neither kind of routing loses much.  Per call in us, 16 /
// 32 rows, even routing and Zipf 1.1 (1.4 at 720):
//                  320            480            560            720            1024           1200
//   N32, layer     126/135 82/86  127/146 95/95  137/150 101/101 145/155 110/101 162/163 137/134 183/175 157/154
//   N32, routed    114/108 63/65  112/115 77/73  122/124 82/79  124/142 87/81  138/145 111/113 151/153 125/123
//   N16, layer     131/138 83/87  132/148 96/95  141/152 102/101 149/159 111/101 165/166 139/134 186/178 159/156
//   N16, routed    119/111 64/65  117/118 79/74  127/128 82/80  129/145 88/80  143/148 112/112 155/155 127/123
// The 64-row tiles before these took, for the routed entries, 115 / 73 us at 320,
// 139 / 93 (N32) and 135 / 93 (N16) at 720 and 167 / 139 at 1200: 16 rows on
// N16 banks at 320 and 32 rows there at 720 would be slower than that on evenly
// routed batches.  N32 routed projections alone at 640-720 tokens are, by 1-2 %.
int grouped_tile_rows(int T) {
    if (kRoutedTile == 32) return T <= 512 ? 16 : 32;
    return T <= 192 || (T > 576 && T <= 1024) ? 16 : 32;
}

hipError_t launch_grouped_mfma(const MfmaArgs& a, bool gateup, int qmax, int T, int max_tiles, hipStream_t s) {
    if (max_tiles <= 0) return hipSuccess;
    // 16-row tiles take eight-wave gate-up blocks (two per CU), 32-row ones
    // four-wave blocks of two passes (two per CU, whose prologue and epilogue
    // overlap the other's stream; eight-wave blocks fit once: 8192 tokens 286
    // -> 331 us).
    //  - up to 64 tokens an expert seldom has a second m-tile, so the codes
    //    are read once and bypass the caches (48 tokens: gate-up 42.5 -> 41.6
    //    us, down 24.4 -> 23.2); beyond, skewed routing re-reads them (512
    //    tokens, Zipf 1.1: 37.6 against 48.6 us) and plain loads are better;
    //  - down blocks cover 256 columns up to 64 tokens, where few experts leave
    //    the chip empty (Zipf 1.1, 256 / 512 / 1024 columns: 33 tokens 8.7 /
    //    10.1 / 13.6 us, 64 tokens 9.8 / 10.9 / 14.3; evenly routed 24.0 / 24.3 /
    //    24.1), 512 beyond (1120 tokens 37 us against 39 with 1024, 64 with
    //    256), and 1024 where every expert has several tiles and staging the rows
    //    half as often counts for more than the extra blocks (even routing, N16
    //    banks, 512 / 1024 columns: 2100 tokens 58.0 / 60.1, 4000 97.0 / 93.8,
    //    8192 191 / 178; Zipf 1.1: 53.8 / 57.3, 91.3 / 95.6, 173.6 / 170.8).
    if (T <= 64) return launch_tiles<16, 8, 4, 1, true>(a, gateup, qmax, max_tiles, s);
    if (grouped_tile_rows(T) == 16) return launch_tiles<16, 8, 4, 2, false>(a, gateup, qmax, max_tiles, s);
    if (T <= 5120) return launch_tiles<32, 4, 4, 2, false>(a, gateup, qmax, max_tiles, s);
    return launch_tiles<32, 4, 4, 4, false>(a, gateup, qmax, max_tiles, s);
}

}  // namespace ornith
