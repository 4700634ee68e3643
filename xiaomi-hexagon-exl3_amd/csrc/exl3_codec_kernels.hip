// exl3_codec_kernels.hip -- gfx950 codec kernels of the EXL3 layer:
//   codebook_kernel    exl3::decode_codebook, bit-exact
//   hadamard_kernel    exl3::hadamard128, bit-exact
//   decode_kernel      trellis tiles -> row-major fp16, bit-exact (exl3::decode_inner);
//   decode_batch_kernel the same for many whole matrices per launch
//   reconstruct_kernel original-basis weights, bit-exact (exl3::reconstruct)
//   get_rows_kernel    GET_ROWS: columns of the original-basis weights (ggml_exl3_get_rows)
//   pack_records_kernel, validate_kernel, zero_kernel
// Reference semantics: src/exl3_codec.cpp, src/exl3-ggml.cpp:19-49.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <type_traits>

#include "exl3_kernel_common.hpp"

namespace exl3k {

// ============================================================== codebook
template <int CB>
__global__ void codebook_kernel(const uint16_t *__restrict__ states, size_t count, uint16_t *__restrict__ out) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) out[i] = codebook_one<CB>(states[i]);
}

hipError_t launch_codebook(const uint16_t *states, size_t count, int cb, uint16_t *out, hipStream_t stream) {
    const dim3 grid((unsigned)((count + 255) / 256)), block(256);
    switch (cb) {
    case 0: codebook_kernel<0><<<grid, block, 0, stream>>>(states, count, out); break;
    case 1: codebook_kernel<1><<<grid, block, 0, stream>>>(states, count, out); break;
    default: codebook_kernel<2><<<grid, block, 0, stream>>>(states, count, out); break;
    }
    return hipGetLastError();
}

// ============================================================== H128
__global__ __launch_bounds__(64) void hadamard_kernel(float *__restrict__ values) {
    __shared__ float v[128];
    float *blk = values + (size_t)blockIdx.x * 128;
    const int t = threadIdx.x;
    v[t] = blk[t];
    v[t + 64] = blk[t + 64];
    __syncthreads();
    h128_lds(v, 1, 128, t, 64);
    blk[t] = v[t];
    blk[t + 64] = v[t + 64];
}

hipError_t launch_hadamard(float *values, size_t count, hipStream_t stream) {
    if (count) hadamard_kernel<<<dim3((unsigned)(count / 128)), dim3(64), 0, stream>>>(values);
    return hipGetLastError();
}

// ============================================================== zero fill
__global__ void zero_kernel(uint32_t *__restrict__ p, size_t words) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < words; i += (size_t)gridDim.x * blockDim.x)
        p[i] = 0u;
}

hipError_t launch_zero(void *ptr, size_t bytes, hipStream_t stream) {
    const size_t words = bytes / 4;
    if (words) {
        const unsigned blocks = (unsigned)((words + 255) / 256 < 4096 ? (words + 255) / 256 : 4096);
        zero_kernel<<<dim3(blocks), dim3(256), 0, stream>>>((uint32_t *)ptr, words);
    }
    return hipGetLastError();
}

// ============================================================== decode
// A unit is one tile row of 8 tiles (16 rows x 128 columns) and belongs to one wave:
// lane 8 t + j decodes chunk j of tile t (decode_chunk: columns j and j + 8 of it, all
// 16 rows, two rows per word).  Neighbouring lanes trade halves (one DPP move and one
// v_perm per word), so that a word is two neighbouring columns of one row, and the wave
// turns the unit in its own LDS rows (272 bytes apart: 4-byte writes and 16-byte reads
// without bank conflicts; no barrier, a wave's LDS accesses stay in order) into
// 256-byte row segments.
// Bound: HBM.  The projections of a layer of hidden 2048 (k / v 512, 6144 wide MLP, 6 / 4
// / 3 bits, 121 MB) in one batch 32.5 -> 23.1 us, 5.3 TB/s where a large copy reaches
// 5.1; against a launch per rate, runs of 16 positions loaded word by word and turned
// through 2-byte LDS writes.  A second unit per wave, its words loaded ahead, 23.9 us;
// four 29.1 (fewer waves in flight).
constexpr int kDecodeRowWords = 68;
template <int K, int CB>
__device__ __forceinline__ void decode_unit(const uint8_t *__restrict__ src, int records_layout, size_t k, size_t n,
                                            size_t rk, size_t block, size_t first_tile, size_t tile_count,
                                            uint16_t *__restrict__ out, uint32_t *rows) {
    const int lane = threadIdx.x & 63, j = lane & 7, odd = j & 1;
    const size_t t0 = block * 8 + (lane >> 3), t = t0 < tile_count ? t0 : tile_count - 1;  // past the end: not stored
    uint32_t w[K];
    load_chunk<K>((const uint8_t *)(tile_ptr<K>(src, records_layout, k, n, rk, first_tile + t) + j * K), w);
    const uint32_t p1 = (uint32_t)__builtin_amdgcn_mov_dpp((int)w[K - 1], 0x121, 0xF, 0xF, false);  // row_ror:1
    const uint32_t p9 = (uint32_t)__builtin_amdgcn_mov_dpp((int)w[K - 1], 0x129, 0xF, 0xF, false);  // row_ror:9
    uint32_t first = j == 0 ? ~0u : 0u;
    asm("" : "+v"(first));  // a mask: v_bfi_b32, not a select on vcc
    u4 fr[4];
    decode_chunk<K, CB>(w, (first & p9) | (~first & p1), fr);
    // words of an even lane: rows 2 v of columns j, j + 1; of an odd one: rows 2 v + 1 of j - 1, j
    const uint32_t sel = odd ? 0x03020706u : 0x05040100u;
    uint32_t *dst = rows + odd * kDecodeRowWords + (lane >> 3) * 8 + (j >> 1);
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        const uint32_t p[4] = {fr[f].x, fr[f].y, fr[f].z, fr[f].w};
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const uint32_t q = (uint32_t)__builtin_amdgcn_mov_dpp((int)p[v], 0xB1, 0xF, 0xF, false);  // lane ^ 1
            dst[(8 * (f & 1) + 2 * v) * kDecodeRowWords + 4 * (f >> 1)] = __builtin_amdgcn_perm(q, p[v], sel);
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const size_t width = tile_count * 16, c0 = block * 128 + (lane & 15) * 8;  // output row length, column
    if (c0 < width) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = 4 * i + (lane >> 4);
            const u4 v = *(const u4 *)(rows + row * kDecodeRowWords + (lane & 15) * 4);
            // streaming store: the fp16 output is written once and not read back here
            __builtin_nontemporal_store(v, (u4 *)(out + (rk * 16 + row) * width + c0));
        }
    }
}

// columns [16 first_tile, + 16 tile_count) of one matrix; grid (column blocks, tile rows)
template <int K, int CB>
__global__ __launch_bounds__(kDecodeWaves * 64) void decode_kernel(const uint8_t *__restrict__ src,
                                                                   int records_layout, size_t k, size_t n,
                                                                   size_t first_tile, size_t tile_count,
                                                                   uint16_t *__restrict__ out) {
    __shared__ __attribute__((aligned(16))) uint32_t turn[kDecodeWaves][16 * kDecodeRowWords];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const size_t block = (size_t)blockIdx.x * kDecodeWaves + wave;
    if (block * 8 < tile_count)  // whole waves, no barrier follows
        decode_unit<K, CB>(src, records_layout, k, n, blockIdx.y, block, first_tile, tile_count, out, turn[wave]);
}

// Several whole matrices, of any rates, in one launch.  Workgroup w belongs to the matrix
// m whose range [wg_begin[m], wg_begin[m + 1]) holds it; its waves take neighbouring units.
template <int K, int CB>
__device__ __forceinline__ void decode_unit_of(const DecodeBatch &batch, int m, int records_layout, uint32_t *rows) {
    const size_t k = batch.k[m], n = batch.n[m];
    const unsigned gx = (unsigned)((n + 127) >> 7);
    const unsigned u = (blockIdx.x - batch.wg_begin[m]) * kDecodeWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned rk = u / gx;
    if (rk < (unsigned)(k >> 4))  // whole waves, no barrier follows
        decode_unit<K, CB>((const uint8_t *)batch.src[m], records_layout, k, n, rk, u - rk * gx, 0, n >> 4,
                           batch.out[m], rows);
}

template <int CB>
__global__ __launch_bounds__(kDecodeWaves * 64) void decode_batch_kernel(DecodeBatch batch, int records_layout) {
    __shared__ __attribute__((aligned(16))) uint32_t turn[kDecodeWaves][16 * kDecodeRowWords];
    const unsigned w = blockIdx.x;
    int m = 0;
    for (int i = 1; i < batch.count; ++i)
        if (w >= batch.wg_begin[i]) m = i;
    uint32_t *rows = turn[threadIdx.x >> 6];
    switch (batch.bits[m]) {
    case 1: decode_unit_of<1, CB>(batch, m, records_layout, rows); break;
    case 2: decode_unit_of<2, CB>(batch, m, records_layout, rows); break;
    case 3: decode_unit_of<3, CB>(batch, m, records_layout, rows); break;
    case 4: decode_unit_of<4, CB>(batch, m, records_layout, rows); break;
    case 5: decode_unit_of<5, CB>(batch, m, records_layout, rows); break;
    case 6: decode_unit_of<6, CB>(batch, m, records_layout, rows); break;
    case 7: decode_unit_of<7, CB>(batch, m, records_layout, rows); break;
    default: decode_unit_of<8, CB>(batch, m, records_layout, rows); break;
    }
}

template <int K>
static hipError_t launch_decode_k(const void *src, int rl, int cb, size_t k, size_t n, size_t first, size_t count,
                                  uint16_t *out, hipStream_t stream) {
    const size_t tiles = count / 16;
    const dim3 grid((unsigned)((tiles + 8 * kDecodeWaves - 1) / (8 * kDecodeWaves)), (unsigned)(k / 16));
    const dim3 block(kDecodeWaves * 64);
    const uint8_t *s = (const uint8_t *)src;
    switch (cb) {
    case 0: decode_kernel<K, 0><<<grid, block, 0, stream>>>(s, rl, k, n, first / 16, tiles, out); break;
    case 1: decode_kernel<K, 1><<<grid, block, 0, stream>>>(s, rl, k, n, first / 16, tiles, out); break;
    default: decode_kernel<K, 2><<<grid, block, 0, stream>>>(s, rl, k, n, first / 16, tiles, out); break;
    }
    return hipGetLastError();
}

hipError_t launch_decode_batch(const DecodeBatch &b, int rl, int cb, unsigned wgs, hipStream_t stream) {
    const dim3 grid(wgs), block(kDecodeWaves * 64);
    switch (cb) {
    case 0: decode_batch_kernel<0><<<grid, block, 0, stream>>>(b, rl); break;
    case 1: decode_batch_kernel<1><<<grid, block, 0, stream>>>(b, rl); break;
    default: decode_batch_kernel<2><<<grid, block, 0, stream>>>(b, rl); break;
    }
    return hipGetLastError();
}

hipError_t launch_decode(const void *src, int rl, int bits, int cb, size_t k, size_t n, size_t first, size_t count,
                         uint16_t *out, hipStream_t stream) {
    switch (bits) {
    case 1: return launch_decode_k<1>(src, rl, cb, k, n, first, count, out, stream);
    case 2: return launch_decode_k<2>(src, rl, cb, k, n, first, count, out, stream);
    case 3: return launch_decode_k<3>(src, rl, cb, k, n, first, count, out, stream);
    case 4: return launch_decode_k<4>(src, rl, cb, k, n, first, count, out, stream);
    case 5: return launch_decode_k<5>(src, rl, cb, k, n, first, count, out, stream);
    case 6: return launch_decode_k<6>(src, rl, cb, k, n, first, count, out, stream);
    case 7: return launch_decode_k<7>(src, rl, cb, k, n, first, count, out, stream);
    default: return launch_decode_k<8>(src, rl, cb, k, n, first, count, out, stream);
    }
}

// ============================================================== reconstruct
// A wave holds one tile row (16 rows x 128 columns, 8 tiles) of a 128-column
// block, decoded a chunk per lane (decode_chunk): lane l, with b =
// h128_lane_block(l % 16), has chunk j = b % 8 of tile tc = b / 8 + 2 (l / 16),
// that is columns 16 tc + j and 16 tc + j + 8, all 16 rows.  Column bits 0, 1, 2, 4
// (strides 1, 2, 4, 16) are then lane bits one DPP read apart (dpp_block_stage8),
// bit 3 is the register, bits 5 and 6 are lane bits 4 and 5.  frag[f] holds rows
// 8 (f % 2) .. + 7 of column 16 tc + j + 8 (f / 2), two rows per word.
template <int K>
__device__ __forceinline__ void load_tile_row(const uint8_t *__restrict__ src, int records_layout, size_t k, size_t n,
                                              size_t rk, size_t cn0, int lane, uint32_t (&w)[K]) {
    const int b = h128_lane_block(lane & 15), tc = (b >> 3) + 2 * (lane >> 4);
    load_chunk<K>((const uint8_t *)(tile_ptr<K>(src, records_layout, k, n, rk, cn0 + tc) + (b & 7) * K), w);
}
template <int K, int CB>
__device__ __forceinline__ void decode_tile_row(const uint32_t (&w)[K], int lane, u4 (&frag)[4]) {
    const int b = h128_lane_block(lane & 15);
    // the previous chunk of the tile (cyclic): the lane holding block (j + 7) % 8
    const int prev_lane = (lane & 48) | h128_lane_block((b & 8) | ((b + 7) & 7));
    const uint32_t prev = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * prev_lane, (int)w[K - 1]);
    decode_chunk<K, CB>(w, prev, frag);
}

// One workgroup of 8 waves per 128x128 block, wave tr its tile row tr.  H128 along
// n stays in the wave: strides 1, 2, 4 and 16 are DPP fmacs, 8 is between registers,
// and 32 and 64 exchange a lane bit with the register bit (permlane swaps), after
// which the butterfly is between registers too.  H128 along k does strides 1..8 in
// registers (a lane has all 16 rows of its columns), goes through LDS once, and does
// 16..64 between the eight values a thread reads back (4 columns of row r of every
// tile row).  Every sum has the operands and the stage order of
// src/exl3_codec.cpp:184-202, then fp16((w * su) * sv): bit-exact.  The DPP stages
// hold sgn times the value (round to nearest is sign-symmetric); the sign goes with
// the 1/sqrt(128) scale as fma(v, +-scale, +0), whose +0 turns a negated exact zero
// into the +0 that the plain butterflies give (no sum of theirs is -0: no codebook
// value is, and x - x is +0).
// Bound: VALU (about 30 per weight, ten of them the decode and its conversion) and
// HBM: k = 2048, n = 6144, 4 bits 106.6 -> 10.9 us (31 MB: 2.9 TB/s), against one
// thread per row, then per column, walking the block through LDS (two of four waves
// idle, 2 x 7 x 64 dependent LDS steps).
template <int K, int CB>
__global__ __launch_bounds__(512) void reconstruct_kernel(const uint8_t *__restrict__ src, int records_layout,
                                                          const uint16_t *__restrict__ su,
                                                          const uint16_t *__restrict__ sv, size_t k, size_t n,
                                                          size_t first_column, size_t count,
                                                          uint16_t *__restrict__ out) {
    constexpr float kScale = 0.08838834764831844055f;
    __shared__ __attribute__((aligned(16))) float blk[8 * 16 * 128];  // [tile row][row][column]
    const int tid = threadIdx.x, lane = tid & 63;
    const int tr = __builtin_amdgcn_readfirstlane(tid >> 6);
    const size_t bc = blockIdx.x, brk = blockIdx.y;  // column block (within the slice), row block
    const size_t gcol0 = first_column + bc * 128;    // absolute column of this block
    u4 frag[4];
    uint32_t w[K];
    load_tile_row<K>(src, records_layout, k, n, brk * 8 + tr, gcol0 / 16, lane, w);
    decode_tile_row<K, CB>(w, lane, frag);
    const int b = h128_lane_block(lane & 15);
    float v[4][8];  // [f][row of the half]
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        const uint32_t p[4] = {frag[f].x, frag[f].y, frag[f].z, frag[f].w};
#pragma unroll
        for (int i = 0; i < 8; ++i) v[f][i] = half_bits_to_float((uint16_t)(p[i >> 1] >> (16 * (i & 1))));
    }
    auto lane_stage = [&](auto sc) {
        constexpr int S = decltype(sc)::value;
        const float sgn = (b & S) ? -1.f : 1.f;
#pragma unroll
        for (int f = 0; f < 4; ++f) dpp_block_stage8<S>(v[f], sgn);
    };
    auto register_stage = [&]() {  // between column halves f and f + 2
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float lo = v[f][i], hi = v[f + 2][i];
                v[f][i] = lo + hi;
                v[f + 2][i] = lo - hi;
            }
    };
    lane_stage(std::integral_constant<int, 1>{});
    lane_stage(std::integral_constant<int, 2>{});
    lane_stage(std::integral_constant<int, 4>{});
    register_stage();                              // stride 8
    lane_stage(std::integral_constant<int, 8>{});  // block bit 3: stride 16
#pragma unroll
    for (int st = 0; st < 2; ++st) {  // strides 32 and 64: the register bit trades places with lane bit 4, then 5
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int x = __float_as_int(v[f][i]), y = __float_as_int(v[f + 2][i]);
                const auto r = st == 0 ? __builtin_amdgcn_permlane16_swap(x, y, false, false)
                                       : __builtin_amdgcn_permlane32_swap(x, y, false, false);
                v[f][i] = __int_as_float(r[0]);
                v[f + 2][i] = __int_as_float(r[1]);
            }
        register_stage();
    }
    const float scale = (__builtin_popcount(b) & 1) ? -kScale : kScale;
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int i = 0; i < 8; ++i) v[f][i] = __builtin_fmaf(v[f][i], scale, 0.f);
    // H128 along k, strides 1, 2, 4 (rows of a half) and 8 (halves)
#pragma unroll
    for (int st = 1; st < 8; st <<= 1)
#pragma unroll
        for (int f = 0; f < 4; ++f)
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (!(i & st)) {
                    const float lo = v[f][i], hi = v[f][i | st];
                    v[f][i] = lo + hi;
                    v[f][i | st] = lo - hi;
                }
#pragma unroll
    for (int f = 0; f < 4; f += 2)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float lo = v[f][i], hi = v[f + 1][i];
            v[f][i] = lo + hi;
            v[f + 1][i] = lo - hi;
        }
    // this lane's column (+ 64 for f >= 2): after the swaps lane bit 4 is column bit 3, lane
    // bit 5 column bit 5 and the register column bit 6; a wave writes 64 columns of one row
    const int col = (b & 7) | ((lane >> 4) & 1) << 3 | (b >> 3) << 4 | (lane >> 5) << 5;
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int i = 0; i < 8; ++i) blk[(tr * 16 + 8 * (f & 1) + i) * 128 + col + 64 * (f >> 1)] = v[f][i];
    // the scales this thread's outputs need: 4 columns, 8 rows
    const int r = tid >> 5, c4 = (tid & 31) * 4;
    const uint8_t *rec = records_layout ? src + ((gcol0 >> 7) * (k >> 7) + brk) * group_bytes(K) : nullptr;
    const uint16_t *su_b = records_layout ? (const uint16_t *)(rec + 2048 * K) : su + brk * 128;
    const uint16_t *sv_b = records_layout ? (const uint16_t *)(rec + 2048 * K + 256) : sv + gcol0;
    float suv[8], svv[4];
#pragma unroll
    for (int t = 0; t < 8; ++t) suv[t] = half_bits_to_float(su_b[16 * t + r]);
#pragma unroll
    for (int c = 0; c < 4; ++c) svv[c] = half_bits_to_float(sv_b[c4 + c]);
    __syncthreads();
    float u[8][4];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const f4 q = *(const f4 *)(blk + (t * 16 + r) * 128 + c4);
        u[t][0] = q.x;
        u[t][1] = q.y;
        u[t][2] = q.z;
        u[t][3] = q.w;
    }
#pragma unroll
    for (int st = 1; st < 8; st <<= 1)  // strides 16, 32, 64
#pragma unroll
        for (int t = 0; t < 8; ++t)
            if (!(t & st))
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const float lo = u[t][c], hi = u[t | st][c];
                    u[t][c] = lo + hi;
                    u[t | st][c] = lo - hi;
                }
    // out is only 2-byte aligned by contract: the hardware takes the 8-byte stores at any alignment
    typedef uint32_t u2_any __attribute__((ext_vector_type(2), aligned(2)));
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        uint32_t h[4];
#pragma unroll
        for (int c = 0; c < 4; ++c)
            h[c] = float_to_half_bits(mul_rn_f32(mul_rn_f32(mul_rn_f32(u[t][c], kScale), suv[t]), svv[c]));
        const u2_any o = {h[0] | h[1] << 16, h[2] | h[3] << 16};
        __builtin_nontemporal_store(o, (u2_any *)(out + (brk * 128 + 16 * t + r) * count + bc * 128 + c4));
    }
}

template <int K>
static hipError_t launch_reconstruct_k(const void *src, int rl, const uint16_t *su, const uint16_t *sv, int cb,
                                       size_t k, size_t n, size_t first, size_t count, uint16_t *out,
                                       hipStream_t stream) {
    const dim3 grid((unsigned)(count / 128), (unsigned)(k / 128)), block(512);
    const uint8_t *s = (const uint8_t *)src;
    switch (cb) {
    case 0: reconstruct_kernel<K, 0><<<grid, block, 0, stream>>>(s, rl, su, sv, k, n, first, count, out); break;
    case 1: reconstruct_kernel<K, 1><<<grid, block, 0, stream>>>(s, rl, su, sv, k, n, first, count, out); break;
    default: reconstruct_kernel<K, 2><<<grid, block, 0, stream>>>(s, rl, su, sv, k, n, first, count, out); break;
    }
    return hipGetLastError();
}

hipError_t launch_reconstruct(const void *src, int rl, const uint16_t *su, const uint16_t *sv, int bits, int cb,
                              size_t k, size_t n, size_t first, size_t count, uint16_t *out, hipStream_t stream) {
    switch (bits) {
    case 1: return launch_reconstruct_k<1>(src, rl, su, sv, cb, k, n, first, count, out, stream);
    case 2: return launch_reconstruct_k<2>(src, rl, su, sv, cb, k, n, first, count, out, stream);
    case 3: return launch_reconstruct_k<3>(src, rl, su, sv, cb, k, n, first, count, out, stream);
    case 4: return launch_reconstruct_k<4>(src, rl, su, sv, cb, k, n, first, count, out, stream);
    case 5: return launch_reconstruct_k<5>(src, rl, su, sv, cb, k, n, first, count, out, stream);
    case 6: return launch_reconstruct_k<6>(src, rl, su, sv, cb, k, n, first, count, out, stream);
    case 7: return launch_reconstruct_k<7>(src, rl, su, sv, cb, k, n, first, count, out, stream);
    default: return launch_reconstruct_k<8>(src, rl, su, sv, cb, k, n, first, count, out, stream);
    }
}

// ============================================================== get_rows
// GET_ROWS on records (src/exl3-ggml.cpp:19-49): out[r][128 kb .. +127] = column
// c = ids[r] % 128 of the original-basis reconstruct of record (ids[r] / 128, kb) as
// a 128x128 matrix, fp16-rounded (then widened for F32 output).  Workgroup (r, kb)
// decodes that record, wave tr its tile row tr (decode_tile_row).
// The H128 over n is restricted to the operations output c depends on (the
// same butterflies in the same order: bit-exact): a stage of stride 2^s keeps
// lo + hi, or lo - hi where bit s of c is set.  Strides 1, 2, 4 and 16 pair lanes, and
// each halves a lane's rows: of two rows A and B the lower lane keeps A's result and
// the upper one B's, so a stage costs two selects, one DPP move and one fma per pair.
// The H128 of the column over k, then fp16((w * su) * sv), are exl3::reconstruct's.
// A stage computes hi' + (+-1) own; where the difference is wanted the lower lane
// holds its negative, and the sign goes with the 1/sqrt(128) scale as
// fma(v, +-scale, +0), as in reconstruct_kernel.
// An id outside [0, n) writes a NaN row and sets *bad_ids (if given) to 1.
// Bound: VALU (about 7 per weight, four of them the decode, and 150 per wave around
// it) and the chain id -> words -> column, hidden only by the four workgroups of a
// CU.  512 ids of a k = 2048, n = 151,936, 6-bit table: 79 -> 32.5 us, against a
// decode into LDS and one thread per row for the H128 over n.  One decode for up to
// eight ids of a column group, counted among 512 ids, is slower: 40.4 us there (5 more
// with the ids fastest in the grid instead of the records), and the ids of a run wait for
// each other (20 equal ids of a 1,024-wide table, 4 bits, 7.1 us against 3.0; 2,048 of a
// 512-wide one, 3 bits, 115 against 30).  It gains 3 to 5 % only where nearly every
// group has eight ids and more (2,048 ids in 64 groups, k = 4096, 3 bits, 205 against 212).
constexpr int kGetRowsThreads = 512;

// One lane-pair stage of two values A, B (rows kept by the lower and the upper lane
// of the pair over block bit S): hi' + al own.  up is all ones on the upper lane: the
// selects are v_bfi_b32, where a select on vcc would be v_cndmask_b32 in its short
// form, which takes 18 cycles a wave here (the others 4).
__device__ __forceinline__ uint32_t pick(uint32_t up, uint32_t a, uint32_t b) { return (up & b) | (~up & a); }
template <int S>
__device__ __forceinline__ float fold_pair(float a, float b, uint32_t up, float al) {
    const uint32_t ai = __float_as_uint(a), bi = __float_as_uint(b);
    const float own = __uint_as_float(pick(up, ai, bi)), send = __uint_as_float(pick(up, bi, ai));
    return __builtin_fmaf(own, al, dpp_block_xor<S>(send));
}

template <int K, int CB>
__global__ __launch_bounds__(kGetRowsThreads) __attribute__((amdgpu_waves_per_eu(8))) void get_rows_kernel(
    const uint8_t *__restrict__ records, size_t k, size_t n, const int32_t *__restrict__ ids, size_t ids_stride,
    size_t count, void *__restrict__ out, int out_f16, size_t out_stride, int *__restrict__ bad_ids) {
    constexpr float kScale = 0.08838834764831844055f;
    __shared__ float colv[128];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // records fastest: the workgroups in flight read whole column groups, each one contiguous
    const size_t r = blockIdx.y + (size_t)gridDim.y * blockIdx.z, kb = blockIdx.x;
    if (r >= count) return;
    const int32_t id = ids[r * ids_stride];
    const size_t o = r * out_stride + kb * 128;
    if (id < 0 || (size_t)id >= n) {
        if (tid < 128) {
            if (out_f16) ((uint16_t *)out)[o + tid] = 0x7e00u;
            else ((uint32_t *)out)[o + tid] = 0x7fc00000u;
        }
        if (tid == 0 && kb == 0 && bad_ids) *bad_ids = 1;
        return;
    }
    const size_t nb = (size_t)id >> 7;
    const int c = id & 127;
    uint32_t w[K];
    load_tile_row<K>(records, 1, k, n, kb * 8 + wave, nb * 8, lane, w);
    const uint8_t *rec = records + (nb * (k >> 7) + kb) * group_bytes(K);
    const uint16_t *su = (const uint16_t *)(rec + 2048 * K);
    const uint16_t sua = su[lane], sub = su[lane + 64];  // for the end, behind the words
    const uint16_t svc = ((const uint16_t *)(rec + 2048 * K + 256))[c];
    u4 frag[4];
    decode_tile_row<K, CB>(w, lane, frag);
    const int b = h128_lane_block(lane & 15);
    uint32_t up1 = (b & 1) ? ~0u : 0u, up2 = (b & 2) ? ~0u : 0u, up4 = (b & 4) ? ~0u : 0u, up8 = (b & 8) ? ~0u : 0u;
    asm("" : "+v"(up1), "+v"(up2), "+v"(up4), "+v"(up8));  // masks, not conditions
    float al[7];
#pragma unroll
    for (int s = 0; s < 7; ++s) al[s] = (c >> s) & 1 ? -1.f : 1.f;
    float t[4][2][2];  // stride 1, on packed row pairs: [f][row pair][row], rows 8 (f % 2) + 4 pair + 2 b0 + row
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int vp = 0; vp < 2; ++vp) {
            const uint32_t lo = vp ? frag[f].z : frag[f].x, hi = vp ? frag[f].w : frag[f].y;
            const uint32_t own = pick(up1, lo, hi);
            const uint32_t got = (uint32_t)__builtin_amdgcn_mov_dpp((int)pick(up1, hi, lo), 0xB1, 0xF, 0xF, false);
#pragma unroll
            for (int h = 0; h < 2; ++h)
                t[f][vp][h] = __builtin_fmaf(half_bits_to_float((uint16_t)(own >> (16 * h))), al[0],
                                             half_bits_to_float((uint16_t)(got >> (16 * h))));
        }
    float e[4][2];  // stride 2: rows 8 (f % 2) + 4 b1 + 2 b0 + row
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int h = 0; h < 2; ++h) e[f][h] = fold_pair<2>(t[f][0][h], t[f][1][h], up2, al[1]);
    float g[2][2];  // stride 4: rows 8 b2 + 4 b1 + 2 b0 + row, column half f / 2
#pragma unroll
    for (int ch = 0; ch < 2; ++ch)
#pragma unroll
        for (int h = 0; h < 2; ++h) g[ch][h] = fold_pair<4>(e[2 * ch][h], e[2 * ch + 1][h], up4, al[2]);
    float a[2];  // stride 8: the column halves
#pragma unroll
    for (int h = 0; h < 2; ++h) a[h] = __builtin_fmaf(g[1][h], al[3], g[0][h]);
    float z = fold_pair<8>(a[0], a[1], up8, al[4]);  // stride 16: row pair split over b3
    {  // strides 32, 64: every lane of the four 16-lane rows ends with the sum
        const auto s32 = __builtin_amdgcn_permlane16_swap(__float_as_int(z), __float_as_int(z), false, false);
        z = __builtin_fmaf(__int_as_float(s32[1]), al[5], __int_as_float(s32[0]));
        const auto s64 = __builtin_amdgcn_permlane32_swap(__float_as_int(z), __float_as_int(z), false, false);
        z = __builtin_fmaf(__int_as_float(s64[1]), al[6], __int_as_float(s64[0]));
    }
    // the lower lane of a pair holds own +- hi negated where the stage subtracts
    const uint32_t neg = ((c & 1) ? ~up1 : 0u) ^ ((c & 2) ? ~up2 : 0u) ^ ((c & 4) ? ~up4 : 0u) ^ ((c & 16) ? ~up8 : 0u);
    const float scale = __uint_as_float(__float_as_uint(kScale) ^ (neg & 0x80000000u));
    // this lane's row of the tile row: block bits 2, 1, 0 and the half of its row pair (bit 3)
    const int row = 16 * wave + (up4 & 8) + (up2 & 4) + (up1 & 2) + (up8 & 1);
    if (lane < 16) colv[row] = __builtin_fmaf(z, scale, 0.f);
    __syncthreads();
    if (wave == 0) {
        float e0 = colv[lane], e1 = colv[lane + 64];
        h128_wave(e0, e1, lane);
        const uint16_t h0 = float_to_half_bits(mul_rn_f32(mul_rn_f32(e0, half_bits_to_float(sua)), half_bits_to_float(svc)));
        const uint16_t h1 = float_to_half_bits(mul_rn_f32(mul_rn_f32(e1, half_bits_to_float(sub)), half_bits_to_float(svc)));
        if (out_f16) {
            ((uint16_t *)out)[o + lane] = h0;
            ((uint16_t *)out)[o + lane + 64] = h1;
        } else {
            ((float *)out)[o + lane] = half_bits_to_float(h0);
            ((float *)out)[o + lane + 64] = half_bits_to_float(h1);
        }
    }
}

template <int K>
static hipError_t launch_get_rows_k(const void *records, int cb, size_t k, size_t n, const int32_t *ids,
                                    size_t ids_stride, size_t count, void *out, int out_f16, size_t out_stride,
                                    int *bad_ids, hipStream_t stream) {
    const size_t gy = count < 65535 ? count : 65535;  // z then stays within 65,535 for any count
    const dim3 grid((unsigned)(k / 128), (unsigned)gy, (unsigned)((count + gy - 1) / gy)), block(kGetRowsThreads);
    const uint8_t *rec = (const uint8_t *)records;
    switch (cb) {
    case 0: get_rows_kernel<K, 0><<<grid, block, 0, stream>>>(rec, k, n, ids, ids_stride, count, out, out_f16,
                                                              out_stride, bad_ids); break;
    case 1: get_rows_kernel<K, 1><<<grid, block, 0, stream>>>(rec, k, n, ids, ids_stride, count, out, out_f16,
                                                              out_stride, bad_ids); break;
    default: get_rows_kernel<K, 2><<<grid, block, 0, stream>>>(rec, k, n, ids, ids_stride, count, out, out_f16,
                                                              out_stride, bad_ids); break;
    }
    return hipGetLastError();
}

hipError_t launch_get_rows(const void *records, int bits, int cb, size_t k, size_t n, const int32_t *ids,
                           size_t ids_stride, size_t count, void *out, int out_f16, size_t out_stride, int *bad_ids,
                           hipStream_t stream) {
    switch (bits) {
    case 1: return launch_get_rows_k<1>(records, cb, k, n, ids, ids_stride, count, out, out_f16, out_stride, bad_ids, stream);
    case 2: return launch_get_rows_k<2>(records, cb, k, n, ids, ids_stride, count, out, out_f16, out_stride, bad_ids, stream);
    case 3: return launch_get_rows_k<3>(records, cb, k, n, ids, ids_stride, count, out, out_f16, out_stride, bad_ids, stream);
    case 4: return launch_get_rows_k<4>(records, cb, k, n, ids, ids_stride, count, out, out_f16, out_stride, bad_ids, stream);
    case 5: return launch_get_rows_k<5>(records, cb, k, n, ids, ids_stride, count, out, out_f16, out_stride, bad_ids, stream);
    case 6: return launch_get_rows_k<6>(records, cb, k, n, ids, ids_stride, count, out, out_f16, out_stride, bad_ids, stream);
    case 7: return launch_get_rows_k<7>(records, cb, k, n, ids, ids_stride, count, out, out_f16, out_stride, bad_ids, stream);
    default: return launch_get_rows_k<8>(records, cb, k, n, ids, ids_stride, count, out, out_f16, out_stride, bad_ids, stream);
    }
}

// ============================================================== records
// One workgroup per record (nb, kb): 64 tiles (tile (r, c) <- upstream tile
// (8 kb + r, 8 nb + c)), then su[128 kb ..], sv[128 nb ..].
__global__ __launch_bounds__(256) void pack_records_kernel(const uint16_t *__restrict__ packed,
                                                           const uint16_t *__restrict__ su,
                                                           const uint16_t *__restrict__ sv, int bits, size_t k,
                                                           size_t n, uint8_t *__restrict__ records) {
    const size_t kbs = k / 128, rec_id = blockIdx.x;
    const size_t nb = rec_id / kbs, kb = rec_id - nb * kbs;
    uint8_t *g = records + rec_id * group_bytes(bits);
    const int tile_u4 = 2 * bits;  // 32*bits bytes per tile = 2*bits uint4
    for (int i = threadIdx.x; i < 64 * tile_u4; i += blockDim.x) {
        const int t = i / tile_u4, o = i - t * tile_u4;
        const size_t up = (kb * 8 + (t >> 3)) * (n / 16) + nb * 8 + (t & 7);
        ((uint4 *)g)[i] = ((const uint4 *)(packed + up * 16 * bits))[o];
    }
    if (threadIdx.x < 16) ((uint4 *)(g + 2048 * bits))[threadIdx.x] = ((const uint4 *)(su + kb * 128))[threadIdx.x];
    else if (threadIdx.x < 32)
        ((uint4 *)(g + 2048 * bits + 256))[threadIdx.x - 16] = ((const uint4 *)(sv + nb * 128))[threadIdx.x - 16];
}

hipError_t launch_pack_records(const uint16_t *packed, const uint16_t *su, const uint16_t *sv, int bits, size_t k,
                               size_t n, void *records, hipStream_t stream) {
    const size_t recs = (k / 128) * (n / 128);
    pack_records_kernel<<<dim3((unsigned)recs), dim3(256), 0, stream>>>(packed, su, sv, bits, k, n,
                                                                         (uint8_t *)records);
    return hipGetLastError();
}

__global__ void set_one_kernel(int *p) { *p = 1; }

// patches/llama-exl3.patch:327-338: a scale is invalid when its exponent field is all ones
__global__ __launch_bounds__(256) void validate_kernel(const uint8_t *__restrict__ records, int bits,
                                                       int *__restrict__ result) {
    const uint16_t *s = (const uint16_t *)(records + (size_t)blockIdx.x * group_bytes(bits) + 2048 * bits);
    if ((s[threadIdx.x] & 0x7c00u) == 0x7c00u) *result = 0;
}

hipError_t launch_validate(const void *records, size_t nrecords, int bits, int *result, hipStream_t stream) {
    set_one_kernel<<<1, 1, 0, stream>>>(result);
    if (nrecords) validate_kernel<<<dim3((unsigned)nrecords), dim3(256), 0, stream>>>((const uint8_t *)records, bits, result);
    return hipGetLastError();
}

}  // namespace exl3k
