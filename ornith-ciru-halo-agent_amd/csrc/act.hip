// Activation preparation: 128-point Hadamard transform + group-256
// quantisation into the int8 layout described in common.hpp.
//   act_bf16   - routed gate / dense input (routed_storage_n32_consumer.cpp:22-76,
//                dense_g256_consumer.cpp:27-73, dense_n32 :276-322)
// One wave owns one (row, 256-group); four waves per block.
#include "kernels.hpp"
#include "timing.hpp"
#include "act.hpp"

namespace ornith {

template <int QMAX>
__global__ __launch_bounds__(256) void act_bf16_kernel(const uint16_t* __restrict__ x, int64_t stride, int rows,
                                                       int groups, const int32_t* __restrict__ ids,
                                                       uint32_t* __restrict__ words, uint16_t* __restrict__ scales,
                                                       int32_t* __restrict__ sums, uint32_t* sticky,
                                                       uint32_t flag_input, uint32_t flag_act) {
    act_bf16_block<QMAX>(int(blockIdx.x), x, stride, rows, groups, ids, words, scales, sums, sticky, flag_input,
                         flag_act);
}

hipError_t launch_act_bf16(const uint16_t* x, int64_t stride, int rows, int K, int qmax, const int32_t* ids,
                           uint32_t* words, uint16_t* scales, int32_t* sums, uint32_t* sticky,
                           uint32_t flag_input, uint32_t flag_act, hipStream_t s) {
    const int groups = K / kGroup;
    const int waves = (rows * groups + 3) / 4;
    const dim3 grid((waves + 3) / 4), block(256);
    if (qmax == 127)
        timed_launch("act", act_bf16_kernel<127>, dim3(grid), dim3(block), 0, s, x, stride, rows, groups, ids, words, scales, sums, sticky,
                                                     flag_input, flag_act);
    else
        timed_launch("act", act_bf16_kernel<7>, dim3(grid), dim3(block), 0, s, x, stride, rows, groups, ids, words, scales, sums, sticky,
                                                   flag_input, flag_act);
    return hipGetLastError();
}

// ---- dense bf16 prefill operands (dense_g256_consumer.cpp:192-229) ----------
// Four packed code words per thread (32 bf16 weights RN(RN(s*code)+off)).
// Threads walk the code words in storage order ([N/tile, K/256, 32, tile]:
// column fastest), four adjacent columns each, so a wave reads one contiguous
// 1 KiB run; each word becomes its column's 16-byte run of eight weights
// (tile / 4 lanes per chunk j, so every row gets 64 / (tile / 4) adjacent
// runs per wave).
__global__ __launch_bounds__(256) void dequantize_bf16_kernel(const uint32_t* __restrict__ codes,
                                                              const uint32_t* __restrict__ meta, int N, int K,
                                                              int tile, uint16_t* __restrict__ w, uint32_t* sticky) {
    const size_t idx = (size_t(blockIdx.x) * 256 + threadIdx.x) * 4;   // first of four words, storage order
    const size_t total = size_t(N) * (K / 8);
    if (idx >= total) return;
    const int groups = K / kGroup;
    const int c = int(idx % tile);                               // columns c .. c+3 of the tile
    const size_t rest = idx / tile;                              // (column tile, group, chunk j)
    const int j = int(rest % 32);
    const size_t tg = rest / 32;                                 // column tile * groups + group
    const int g = int(tg % groups), nt = int(tg / groups);
    const int kw = g * 32 + j;
    // codes and metadata carry 4-byte alignment only (prepare_bf16's contract)
    const uint32_t* cp = codes + idx;
    const uint32_t* mp = meta + tg * tile + c;
    const uint32_t wv[4] = {cp[0], cp[1], cp[2], cp[3]}, mv[4] = {mp[0], mp[1], mp[2], mp[3]};
    uint32_t flags = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float scale = f16_bits_to_f32(mv[e] & 0xffffu), offset = f16_bits_to_f32(mv[e] >> 16);
        uint32_t out[4];
#pragma unroll
        for (int i = 0; i < 8; i += 2) {
            const float a = scale * float((wv[e] >> (4 * i)) & 15u) + offset;
            const float b = scale * float((wv[e] >> (4 * i + 4)) & 15u) + offset;
            const uint16_t ra = f32_to_bf16_bits(a), rb = f32_to_bf16_bits(b);
            if ((ra & 0x7f80u) == 0x7f80u || (rb & 0x7f80u) == 0x7f80u) flags |= kDenseNonfiniteBf16;
            out[i / 2] = ra | (uint32_t(rb) << 16);
        }
        const int n = nt * tile + c + e;
        *reinterpret_cast<uint4*>(w + size_t(n) * K + size_t(kw) * 8) = make_uint4(out[0], out[1], out[2], out[3]);
    }
    flag_or(sticky, flags);
}

hipError_t launch_dequantize_bf16(const uint32_t* codes, const uint32_t* meta, int N, int K, int tile, uint16_t* w,
                                  uint32_t* sticky, hipStream_t s) {
    const size_t threads = size_t(N) * (K / 8) / 4;    // tile >= 16: four words never straddle a tile row
    timed_launch("dequantize", dequantize_bf16_kernel, dim3((threads + 255) / 256), dim3(256), 0, s, codes, meta, N, K, tile, w, sticky);
    return hipGetLastError();
}

__global__ void fill_u32_kernel(uint32_t* p, size_t n, uint32_t v) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

hipError_t launch_fill_u32(uint32_t* p, size_t n, uint32_t v, hipStream_t s) {
    if (!n) return hipSuccess;
    timed_launch("fill", fill_u32_kernel, dim3((n + 255) / 256), dim3(256), 0, s, p, n, v);
    return hipGetLastError();
}

}  // namespace ornith
