// INT8 attention of single tokens, verify blocks and small prefill chunks over the KV cache.
//
// Three entry points:
//   * the reference's three-kernel reader (kernels.metal:147-156,163-166):
//     batch_attention_scores_int8 -> attention_softmax -> batch_attention_values_int8,
//     FP32 scores in a caller buffer; serves callers that dispatch it as the
//     reference does (QwenEngine.cs:161-165, Prefill.cs:280-285) and verify blocks
//     of more than 64 rows.
//   * attention_decode_int8: one fused split-K pass that streams the INT8 K/V
//     pages from HBM once, as whole K rows and whole 128-byte V page-row lines
//     staged through LDS. Scores run on INT8 MFMA straight from the K codes:
//     the FP32 query of each head is split into three INT8 parts,
//     q ~= s_q (q1 + q2 / 254 + q3 / 254^2) with s_q = max|q| / 127 (error
//     <= 6.1e-8 max|q| per element, below the FP32 reader's own summation error),
//     in two MFMAs whose 16 columns are 8 heads x {q1, q2} and 8 heads x q3. PV runs on FP16 MFMA
//     with V codes dequantized exactly in registers and the scaled
//     probabilities 2^7 p*vs[t]/vs_ref (vs_ref = the largest V scale of the split; p is
//     at most 2^8 against a lagging running maximum, so they lie in [0, 2^15]) split
//     into FP16 hi + lo. Scales are applied to scores and probabilities as the
//     reference does (score = dot * ks[t] / 16, P = p * vs[t]).
//   * attention_verify_int8: the same arithmetic for the rows of a verify block, several
//     rows per work-group (rows_int8_kernel).
#include "common.h"
#include <type_traits>
#include "kvmath.h"
#include "mfma.h"

namespace boot {


namespace {

// ---------------------------------------------------------------- reference-compatible reader

// scores[(row*16+h)*K + t] = (q . code) * ks[t*2+h/8] * (1/16), -inf beyond row's causal end
// (kernels.metal:147-152), on INT8 MFMA (v_mfma_i32_16x16x64_i8). Each (row, head) query is split
// into three INT8 parts, q ~= s_q (q1 + q2 / 254 + q3 / 254^2) with s_q = max|q| / 127 (error
// <= 6.1e-8 max|q| per element), the dot products with the codes are exact integers, and their
// combination is FP32 per element: a row's scores do not depend on the rows it is dispatched
// with. Work-group (span = 256 or 512 tokens, KV group, kRows rows): the query operands of its rows
// in LDS (16 columns: 8 heads x {q1, q2}, and 8 heads x q3 twice), wave w takes the span's quarter
// w in pairs of 16-token tiles; each K operand (16 bytes of a token's row per lane) feeds 2 kRows
// MFMAs.
template <int kRows>
__global__ __launch_bounds__(256) void scores_int8_kernel(const float *__restrict__ q, const int8_t *__restrict__ k,
                                                          float *__restrict__ scores, const float *__restrict__ ks,
                                                          uint32_t rows, uint32_t K, uint32_t pos, uint32_t tiles,
                                                          uint32_t zs, uint32_t span) {
    typedef int v4i __attribute__((ext_vector_type(4)));
    __shared__ v4i qop[kRows][2][4][64];   // [row][set][64-dimension step][lane]
    __shared__ float qscale[kRows][8];
    // blocks are dealt to the XCDs round-robin by index: the row blocks of one (tile, group) pair
    // are 8 apart, on one XCD at about the same time, so that the K tile they share comes from HBM once
    const uint32_t xcd = blockIdx.x % 8, j = blockIdx.x / 8, pair = (j / zs) * 8 + xcd;
    if (pair >= 2 * tiles) return;   // padding of the grid to whole rounds of 8
    const uint32_t kt = pair / 2, g = pair % 2, r0 = (j % zs) * kRows;
    const uint32_t nr = min((uint32_t)kRows, rows - r0);
    const uint32_t length = min(pos + rows, K);   // the cache rows read (validated by the launcher)
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = lane & 15, qq = lane >> 4;
    // ---- query parts: thread T takes head T / 32, dimensions 8 (T % 32) .. + 7 of each row
    {
        const int h = tid >> 5, d0 = 8 * (tid & 31);
        auto code = [](float x) { return (uint32_t)(uint8_t)(int8_t)(int)fminf(fmaxf(x, -127.0f), 127.0f); };
#pragma unroll
        for (int r = 0; r < kRows; r++) {
            float x[8];
            const float *src = q + (size_t)(r0 + min((uint32_t)r, nr - 1)) * 4096 + (g * 8 + h) * 256 + d0;
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = src[e];   // (the query binding needs only 4-byte alignment)
            float amax = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(x[e]));
#pragma unroll
            for (int o = 16; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));   // the head's 32 lanes
            const float inv = amax > 0.0f ? 127.0f / amax : 0.0f;
            if ((tid & 31) == 0) qscale[r][h] = amax * (1.0f / 127.0f);
            uint32_t w1[2] = {0, 0}, w2[2] = {0, 0}, w3[2] = {0, 0};
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float z = x[e] * inv, q1 = rintf(z), r1 = z - q1;
                const float q2 = rintf(r1 * 254.0f);
                const float r2 = fmaf(r1, 254.0f, -q2);
                const float q3 = rintf(r2 * 254.0f);
                w1[e >> 2] |= code(q1) << (8 * (e & 3));
                w2[e >> 2] |= code(q2) << (8 * (e & 3));
                w3[e >> 2] |= code(q3) << (8 * (e & 3));
            }
            // dimension d0 + e is byte (d0 % 16) + e of lane 16 ((d0 % 64) / 16) + column of step d0 / 64
            const int step = d0 >> 6, at = 16 * ((d0 & 63) >> 4), half = (d0 & 15) >> 3;
            unsigned char *base = reinterpret_cast<unsigned char *>(&qop[r][0][step][0]);
            *reinterpret_cast<uint2 *>(base + (at + h) * 16 + 8 * half) = make_uint2(w1[0], w1[1]);
            *reinterpret_cast<uint2 *>(base + (at + h + 8) * 16 + 8 * half) = make_uint2(w2[0], w2[1]);
            unsigned char *base3 = reinterpret_cast<unsigned char *>(&qop[r][1][step][0]);
            *reinterpret_cast<uint2 *>(base3 + (at + h) * 16 + 8 * half) = make_uint2(w3[0], w3[1]);
            *reinterpret_cast<uint2 *>(base3 + (at + h + 8) * 16 + 8 * half) = make_uint2(w3[0], w3[1]);
        }
    }
    __syncthreads();
    const bool lo_col = n >= 8;
    // Two 16-token tiles at a time: after the hi/lo exchange lanes n < 8 finish the first and lanes
    // n >= 8 the second, so that one store instruction writes 128 contiguous bytes of each head's row
    // with every lane active. The work-group's `span` tokens (256 or 512) are split over the waves.
    const uint32_t per_wave = span / 4;
#pragma unroll 1
    for (uint32_t tp = 0; tp < per_wave / 32; tp++) {
        const uint32_t ta = kt * span + per_wave * wave + 32 * tp;
        if (ta >= K) break;   // wave-uniform
        v4i kop[2][4];
        float kss[2][4];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const uint32_t tk = min(ta + 16 * u + n, length - 1);   // the lane's K row (an existing one)
#pragma unroll
            for (int jj = 0; jj < 4; jj++)
                kop[u][jj] = *reinterpret_cast<const v4i *>(k + ((size_t)tk * 2 + g) * 256 + 64 * jj + 16 * qq);
#pragma unroll
            for (int i = 0; i < 4; i++) kss[u][i] = ks[(size_t)min(ta + 16 * u + 4 * qq + i, length - 1) * 2 + g];
        }
        const uint32_t tb = ta + (lo_col ? 16 : 0);   // the tile this lane finishes
#pragma unroll
        for (int r = 0; r < kRows; r++) {
            if ((uint32_t)r >= nr) break;   // uniform
            v4i acc[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}}, acc3[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
            for (int u = 0; u < 2; u++)
#pragma unroll
                for (int jj = 0; jj < 4; jj++) {
                    acc[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(kop[u][jj], qop[r][0][jj][lane], acc[u], 0, 0, 0);
                    acc3[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(kop[u][jj], qop[r][1][jj][lane], acc3[u], 0, 0, 0);
                }
            // column n holds head n % 8's part q1 (n < 8) or q2 (n >= 8), both columns its q3; token
            // tb + 4qq + i of this lane's tile
            const float qsc = qscale[r][n & 7];
            const uint32_t last = pos + r0 + r;   // the row's last visible key
            float *dst = scores + ((size_t)(r0 + r) * 16 + g * 8 + (n & 7)) * K;
            float out[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int ma = acc[0][i], oa = __shfl_xor(ma, 8, 64);
                const int mb = acc[1][i], ob = __shfl_xor(mb, 8, 64);
                const float hi = (float)(lo_col ? ob : ma), lo = (float)(lo_col ? mb : oa);
                const int c3 = lo_col ? acc3[1][i] : acc3[0][i];
                const float full = fmaf((float)c3, 1.0f / 64516.0f, fmaf(lo, 1.0f / 254.0f, hi)) * qsc;
                const uint32_t t = tb + 4 * qq + i;
                out[i] = t <= last ? full * (lo_col ? kss[1][i] : kss[0][i]) * (1.0f / 16.0f) : -INFINITY;
            }
            // the lane's four consecutive tokens as one 16-byte store where the row allows it
            const uint32_t t4 = tb + 4 * qq;
            if (t4 + 3 < K && (reinterpret_cast<uintptr_t>(dst + t4) & 15) == 0) {
                *reinterpret_cast<float4 *>(dst + t4) = make_float4(out[0], out[1], out[2], out[3]);
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (t4 + i < K) dst[t4 + i] = out[i];
            }
        }
    }
}

__device__ inline float block_reduce_256(float v, float *partial, bool is_max) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        float other = __shfl_xor(v, o, 64);
        v = is_max ? fmaxf(v, other) : v + other;
    }
    __syncthreads();
    if ((threadIdx.x & 63) == 0) partial[threadIdx.x >> 6] = v;
    __syncthreads();
    float r = partial[0];
    for (int i = 1; i < 4; i++) r = is_max ? fmaxf(r, partial[i]) : r + partial[i];
    return r;
}

// In-place softmax over i <= pos of each row of stride K (kernels.metal:163-166), in two passes
// over chunks of kSoftmaxChunk elements (absolute boundaries, so that a row's result does not
// depend on how many rows the dispatch holds): the chunk's maximum and its sum of exp(x - max),
// then, per chunk, the row's maximum M and sum L merged from those in chunk order and
// x = exp(x - M) / L. Elements past pos are left as they are.
constexpr int kSoftmaxChunk = 8192;
constexpr int kSoftmaxPer = kSoftmaxChunk / 256;

__global__ __launch_bounds__(256) void softmax_stats_kernel(const float *__restrict__ x, float2 *__restrict__ stats,
                                                            uint32_t K, uint32_t pos, uint32_t chunks) {
    __shared__ float partial[4];
    const uint32_t c = blockIdx.x, r = blockIdx.y;
    const float *row = x + (size_t)r * K;
    const uint32_t lo = c * kSoftmaxChunk, hi = min(pos + 1, lo + kSoftmaxChunk);
    // every chunk holds at least one element at or below pos: loads of a clamped index, then the
    // elements past the row's end are masked (no branch per load)
    float e[kSoftmaxPer];
#pragma unroll
    for (int j = 0; j < kSoftmaxPer; j++) e[j] = row[min(lo + threadIdx.x + 256 * j, hi - 1)];
#pragma unroll
    for (int j = 0; j < kSoftmaxPer; j++)
        if (lo + threadIdx.x + 256 * j >= hi) e[j] = -INFINITY;
    float top = -INFINITY;
#pragma unroll
    for (int j = 0; j < kSoftmaxPer; j++) top = fmaxf(top, e[j]);
    top = block_reduce_256(top, partial, true);
    float sum = 0.0f;
    if (top != -INFINITY)
#pragma unroll
        for (int j = 0; j < kSoftmaxPer; j++) sum += expf(e[j] - top);
    sum = block_reduce_256(sum, partial, false);
    if (threadIdx.x == 0) stats[(size_t)r * chunks + c] = make_float2(top, sum);
}

__global__ __launch_bounds__(256) void softmax_apply_kernel(float *__restrict__ x, const float2 *__restrict__ stats,
                                                            uint32_t K, uint32_t pos, uint32_t chunks) {
    const uint32_t c = blockIdx.x, r = blockIdx.y;
    // the chunk's loads go out first; the row's statistics (the same for the whole work-group)
    // are merged while they are in flight
    float *row = x + (size_t)r * K;
    const uint32_t lo = c * kSoftmaxChunk, hi = min(pos + 1, lo + kSoftmaxChunk);
    float e[kSoftmaxPer];
#pragma unroll
    for (int j = 0; j < kSoftmaxPer; j++) e[j] = row[min(lo + threadIdx.x + 256 * j, hi - 1)];
    const float2 *st = stats + (size_t)r * chunks;
    float top = -INFINITY;
    for (uint32_t k = 0; k < chunks; k++) top = fmaxf(top, st[k].x);
    float sum = 0.0f;
    for (uint32_t k = 0; k < chunks; k++)
        if (st[k].x != -INFINITY) sum += st[k].y * expf(st[k].x - top);
    if (hi == lo + kSoftmaxChunk) {   // a whole chunk: no mask per store
#pragma unroll
        for (int j = 0; j < kSoftmaxPer; j++) row[lo + threadIdx.x + 256 * j] = expf(e[j] - top) / sum;
    } else {
#pragma unroll
        for (int j = 0; j < kSoftmaxPer; j++) {
            const uint32_t i = lo + threadIdx.x + 256 * j;
            if (i < hi) row[i] = expf(e[j] - top) / sum;
        }
    }
}

// y[(row*16+h)*256+d] = sum_{t <= pos+row} scores*vs*vcode * sigmoid(gate) (kernels.metal:153-156),
// split over absolute kValuesSplit-token ranges (a row's sum does not depend on the dispatch's
// row count); values_combine_kernel adds the splits in order and applies the gate.
constexpr int kValuesSplit = 512;

// Work-group (split, KV group, kRows rows): O^T[d][c] += V^T[d][t] B[t][c] on
// v_mfma_f32_16x16x16_f16 with the codes exact in FP16 and, per row, B = p * vs * 2^15 / vs_r in
// the 16 columns 8 heads x {FP16 hi, FP16 lo} (vs_r the row's largest V scale over its tokens of
// the split, so that B <= 2^15; hi + lo keeps about 22 bits), the result times vs_r / 2^15. The
// factor 2^15 keeps the probabilities of a long, flat row (p ~ 1 / K) out of FP16's subnormals
// (below 2^-14), where hi and lo would keep only a few bits. Eight waves, wave w taking
// dimensions 32w .. 32w + 31 (96 registers: two work-groups per CU; four waves with 64 dimensions
// each held 168, three per CU, 21.5 against 18.9 us at 4 rows over 30000 keys); a 64-token block
// is four k-steps, lane (n, qq) of step s holding tokens 16qq + 4s .. + 3 of the block for both
// operands (one 16-byte code load per dimension tile covers its four steps), and the next block's
// loads are issued before the current block is staged. Every quantity of a row depends on that
// row's range only, whatever kRows is.
constexpr int kVmBlock = 64;
constexpr float kValuesScale = 32768.0f;   // 2^15: B's factor

template <int kRows>
__global__ __launch_bounds__(512) void values_partial_kernel(const float *__restrict__ scores,
                                                             const int8_t *__restrict__ v, const float *__restrict__ vs,
                                                             float *__restrict__ partial, uint32_t rows, uint32_t K,
                                                             uint32_t pos, uint32_t splits, uint32_t zs) {
    typedef _Float16 half4 __attribute__((ext_vector_type(4)));
    constexpr int kWaves = 8;                           // wave w: dimensions 32w .. 32w + 31
    // B operands [row][k-step][slot]: lane L's operand in slot L ^ ((L / 16) % 4 * 2), each k-step row
    // padded by one slot. A staging store writes one (row, head)'s 64 tokens, which fall in 16
    // slots (4 k-steps x 4 token blocks); without the padding and the XOR the four k-steps (512 bytes
    // apart) and token blocks 0 and 2 share their banks, 8 to 16 lanes per bank; with them the 16
    // slots cover 32 banks. The operand reads (64 slots of one k-step row) stay conflict-free.
    __shared__ uint2 bs[kRows][4][65];
    auto bslot = [](int L) __attribute__((always_inline)) { return L ^ ((L >> 3) & 6); };
    __shared__ float vred[kWaves][kRows];
    // the row blocks of one (split, group) pair 8 blocks apart: one XCD reads the pair's V once
    const uint32_t xcd = blockIdx.x % 8, jb = blockIdx.x / 8, pair = (jb / zs) * 8 + xcd;
    if (pair >= 2 * splits) return;   // padding of the grid to whole rounds of 8
    const uint32_t split = pair / 2, g = pair % 2, r0 = (jb % zs) * kRows;
    const uint32_t nr = min((uint32_t)kRows, rows - r0);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = lane & 15, qq = lane >> 4;
    const uint32_t t0 = split * kValuesSplit;
    const uint32_t t1 = min(pos + r0 + nr, t0 + kValuesSplit);   // the work-group's last row's end
    // each row's largest V scale over its tokens of the split
    float vr[kRows];
    {
        float vm[kRows];
#pragma unroll
        for (int r = 0; r < kRows; r++) vm[r] = 0.0f;
        if (t0 < t1)
#pragma unroll
            for (int k = 0; k < kValuesSplit / 512; k++) {
                const uint32_t t = t0 + tid + 512 * k;
                const float x = vs[(size_t)min(t, t1 - 1) * 2 + g];
#pragma unroll
                for (int r = 0; r < kRows; r++)
                    if (t < pos + r0 + r + 1) vm[r] = fmaxf(vm[r], x);
            }
#pragma unroll
        for (int r = 0; r < kRows; r++) {
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) vm[r] = fmaxf(vm[r], __shfl_xor(vm[r], o, 64));
            if (lane == 0) vred[wave][r] = vm[r];
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kRows; r++) {
            vr[r] = vred[0][r];
#pragma unroll
            for (int w = 1; w < kWaves; w++) vr[r] = fmaxf(vr[r], vred[w][r]);
        }
    }
    floatx4 acc[2][kRows];
#pragma unroll
    for (int dt = 0; dt < 2; dt++)
#pragma unroll
        for (int r = 0; r < kRows; r++) acc[dt][r] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    // staging: thread T takes token T % 64 of the block for row i, head T / 64 (the wave: uniform) of
    // every row i, so that a wave's score loads read 64 consecutive tokens of one (row, head). The
    // loads are unconditional (row and token clamped into the rows and keys that exist) and the
    // causal mask a select at staging time (a select at the load would wait for it there), so no
    // load sits under a per-lane branch.
    const int tok = tid & 63, sh = __builtin_amdgcn_readfirstlane(tid >> 6);
    struct Loads {
        float sc[kRows], sv;
        uint4 w4[2];   // the wave's two dimension tiles: dimension 32 wave + 16 dt + n, tokens 16 qq .. + 15
    };
    auto load = [&](Loads &L, uint32_t tb) __attribute__((always_inline)) {
        const uint32_t t = tb + tok, tc = min(t, t1 - 1);
        L.sv = vs[(size_t)tc * 2 + g];
#pragma unroll
        for (int i = 0; i < kRows; i++) {
            const uint32_t rc = min((uint32_t)i, nr - 1);
            L.sc[i] = scores[((size_t)(r0 + rc) * 16 + g * 8 + sh) * K + tc];
        }
#pragma unroll
        for (int dt = 0; dt < 2; dt++)
            L.w4[dt] = *reinterpret_cast<const uint4 *>(v + value_index((uint64_t)tb * 2 + g, 32 * wave + 16 * dt + n) + 16 * qq);
    };
    Loads cur, nxt;
    if (t0 < t1) load(cur, t0);
    for (uint32_t tb = t0; tb < t1; tb += kVmBlock) {
        const bool more = tb + kVmBlock < t1;   // work-group-uniform
        if (more) load(nxt, tb + kVmBlock);
        __syncthreads();   // the previous block's B reads are done
        {
            // token tok of the block is k = 4 (tok / 16) + tok % 4 of step (tok % 16) / 4: half tok % 4
            // of lane 16 (tok / 16) + column
            const int s = (tok & 15) >> 2, j = tok & 3, lrow = 16 * (tok >> 4);
#pragma unroll
            for (int i = 0; i < kRows; i++) {
                if ((uint32_t)i < nr) {   // uniform
                    const float inv = vr[i] > 0.0f ? kValuesScale / vr[i] : 0.0f;
                    const float p = tb + tok < pos + r0 + i + 1 ? cur.sc[i] : 0.0f;   // the causal mask
                    const float x = p * cur.sv * inv;
                    const _Float16 hi = (_Float16)x, lo = (_Float16)(x - (float)hi);
                    reinterpret_cast<_Float16 *>(&bs[i][s][bslot(lrow + sh)])[j] = hi;
                    reinterpret_cast<_Float16 *>(&bs[i][s][bslot(lrow + sh + 8)])[j] = lo;
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < 4; s++) {
            half4 a[2];
#pragma unroll
            for (int dt = 0; dt < 2; dt++) {
                const uint4 &w = cur.w4[dt];
                const uint32_t word = s == 0 ? w.x : s == 1 ? w.y : s == 2 ? w.z : w.w;
                uint32_t h0, h1;
                i8x4_to_f16(word, h0, h1);
                a[dt] = __builtin_bit_cast(half4, make_uint2(h0, h1));
            }
#pragma unroll
            for (int r = 0; r < kRows; r++) {
                if ((uint32_t)r >= nr) break;   // uniform
                const half4 b = __builtin_bit_cast(half4, bs[r][s][bslot(lane)]);
#pragma unroll
                for (int dt = 0; dt < 2; dt++) acc[dt][r] = __builtin_amdgcn_mfma_f32_16x16x16f16(a[dt], b, acc[dt][r], 0, 0, 0);
            }
        }
        if (more) cur = nxt;
    }
    // the lo column n + 8 joins the hi column n (head n); lanes n < 8 write dimensions 32 wave + 16 dt + 4 qq + e
#pragma unroll
    for (int r = 0; r < kRows; r++) {
        if ((uint32_t)r >= nr) break;
        float *out = partial + (((size_t)(r0 + r) * 2 + g) * splits + split) * 2048;
        const float f = vr[r] * (1.0f / kValuesScale);   // exact: a power of two
#pragma unroll
        for (int dt = 0; dt < 2; dt++) {
            float4 o4;
            o4.x = (acc[dt][r][0] + __shfl_xor(acc[dt][r][0], 8, 64)) * f;
            o4.y = (acc[dt][r][1] + __shfl_xor(acc[dt][r][1], 8, 64)) * f;
            o4.z = (acc[dt][r][2] + __shfl_xor(acc[dt][r][2], 8, 64)) * f;
            o4.w = (acc[dt][r][3] + __shfl_xor(acc[dt][r][3], 8, 64)) * f;
            if (n < 8) *reinterpret_cast<float4 *>(out + n * 256 + 32 * wave + 16 * dt + 4 * qq) = o4;
        }
    }
}

__global__ __launch_bounds__(64) void values_combine_kernel(const float *__restrict__ partial,
                                                             const float *__restrict__ gate, float *__restrict__ y,
                                                             uint32_t splits) {
    const uint32_t h = blockIdx.x / 4, row = blockIdx.y, g = h / 8, d = 64 * (blockIdx.x % 4) + threadIdx.x;
    const float *src = partial + ((size_t)row * 2 + g) * splits * 2048 + (h % 8) * 256 + d;
    float sum = 0.0f;
    for (uint32_t s = 0; s < splits; s += 32) {   // 32 loads in flight, added in split order
        float x[32];
#pragma unroll
        for (int u = 0; u < 32; u++) x[u] = src[(size_t)min(s + u, splits - 1) * 2048];
#pragma unroll
        for (int u = 0; u < 32; u++)
            if (s + u < splits) sum += x[u];
    }
    const size_t i = ((size_t)row * 16 + h) * 256 + d;
    y[i] = sum * (1.0f / (1.0f + expf(-gate[i])));
}

// ---------------------------------------------------------------- fused split-K decode

constexpr int kChunk = 128;                      // tokens per LDS chunk (one 128-byte line per V page row)
constexpr int kDecodeWaves = 8;
constexpr int kMaxSplitTokens = 2048;            // tokens per work-group at most (LDS scales)
constexpr int kPartialFloats = 8 * 256 + 16;    // O[8][256], m[8], l[8] per (row, group, split)
constexpr int kMaxDecodeSplits = 1024;
constexpr float kLog2e = 1.4426950408889634f;

struct DecodeParams {
    const float *q;              // FP32 [rows][16][256] (or qh below)
    const int8_t *k;
    const int8_t *v;
    const float *ks;
    const float *vs;
    const float *gate;
    float *y;
    float *partial;
    uint32_t rows, pos, splits;
    uint32_t split_chunks;   // 128-token chunks per split
    // attention_decode_append_int8 (one row): q is the unrotated query; the kernel rotates it
    // (writing it to `rotated`), quantizes the new token's K (rotated) and V into the cache at
    // `pos` (k_out, v_out, ks_out, vs_out alias k, v, ks, vs) and attends over it
    uint32_t append;
    RopeFreq freq;
    const float *knew, *vnew;    // FP32 [2][256] each
    float *rotated;              // FP32 [16][256]
    int8_t *k_out, *v_out;
    float *ks_out, *vs_out;
    const _Float16 *qh;          // prefill chunks routed here: the grouped FP16 query [2][rows][8][256]
};

// x of lane l ^ 16 (v_permlane16_swap) and of lane l ^ 32 (v_permlane32_swap) added or maxed in:
// with both operands holding x, every lane ends with its own value in one register and its
// partner's in the other; the no-ops cover the cross-lane move's wait states. Registers, not an
// LDS round trip as a shuffle takes.
__device__ inline float xl_sum16(float x) {
    float a = x, b = x;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    return a + b;
}
__device__ inline float xl_sum32(float x) {
    float a = x, b = x;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    return a + b;
}
__device__ inline float xl_max16(float x) {
    float a = x, b = x;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    return fmaxf(a, b);
}
__device__ inline float xl_max32(float x) {
    float a = x, b = x;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    return fmaxf(a, b);
}
// Every element's maximum over the wave: rotations of the 16-lane rows by DPP (the steps of
// several elements interleave, covering each other's wait states), then across the rows
template <int N>
__device__ inline void wave_allmax(float (&x)[N]) {
#pragma unroll
    for (int step = 0; step < 4; step++)
#pragma unroll
        for (int i = 0; i < N; i++) {
            if (step == 0) asm volatile("s_nop 1\n\tv_max_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf" : "+v"(x[i]));
            if (step == 1) asm volatile("s_nop 1\n\tv_max_f32_dpp %0, %0, %0 row_ror:4 row_mask:0xf bank_mask:0xf" : "+v"(x[i]));
            if (step == 2) asm volatile("s_nop 1\n\tv_max_f32_dpp %0, %0, %0 row_ror:2 row_mask:0xf bank_mask:0xf" : "+v"(x[i]));
            if (step == 3) asm volatile("s_nop 1\n\tv_max_f32_dpp %0, %0, %0 row_ror:1 row_mask:0xf bank_mask:0xf" : "+v"(x[i]));
        }
#pragma unroll
    for (int i = 0; i < N; i++) x[i] = xl_max32(xl_max16(x[i]));
}

// sigmoid(x) = 1 / (1 + 2^(-x log2(e))) with the hardware exponential and reciprocal (about an ulp
// each), as the prefill kernels compute it
__device__ inline float sigmoidf(float x) {
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-x * 1.4426950408889634f));
}

// x + x of lane l ^ 8 (the same position in the other half of its 16-lane row) for
// the eight values of two accumulators: one DPP add each, as inline assembly (the DPP
// move builtin was mis-scheduled here, and a cross-lane shuffle costs an LDS round
// trip per value). The sources are MFMA results whose wait states the caller has
// covered and no add reads another's result, so only the block's ends need wait
// states (a register copy the compiler places just before the block).
__device__ inline void add_row_partner8(floatx4 &a, floatx4 &b) {
    float r0, r1, r2, r3, r4, r5, r6, r7;
    asm volatile(
        "s_nop 1\n\t"
        "v_add_f32_dpp %0, %8, %8 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %1, %9, %9 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %2, %10, %10 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %3, %11, %11 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %4, %12, %12 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %5, %13, %13 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %6, %14, %14 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %7, %15, %15 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1"
        : "=&v"(r0), "=&v"(r1), "=&v"(r2), "=&v"(r3), "=&v"(r4), "=&v"(r5), "=&v"(r6), "=&v"(r7)
        : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]));
    a = floatx4{r0, r1, r2, r3};
    b = floatx4{r4, r5, r6, r7};
}

// The same for four integers (MFMA results scaled by ordinary VALU instructions)
__device__ inline void add_row_partner8(int (&a)[4]) {
    int r0, r1, r2, r3;
    asm volatile(
        "s_nop 1\n\t"
        "v_add_u32_dpp %0, %4, %4 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_u32_dpp %1, %5, %5 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_u32_dpp %2, %6, %6 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_u32_dpp %3, %7, %7 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1"
        : "=&v"(r0), "=&v"(r1), "=&v"(r2), "=&v"(r3)
        : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]));
    a[0] = r0;
    a[1] = r1;
    a[2] = r2;
    a[3] = r3;
}

// The largest magnitude of heads whose four dimensions a lane holds, NaN for a head with a NaN (the
// maximum instructions drop it)
template <int N>
__device__ __attribute__((always_inline)) inline void head_max(const float4 (&q)[N], float (&amax)[N]) {
#pragma unroll
    for (int i = 0; i < N; i++) amax[i] = fmaxf(fmaxf(fabsf(q[i].x), fabsf(q[i].y)), fmaxf(fabsf(q[i].z), fabsf(q[i].w)));
    wave_allmax(amax);
#pragma unroll
    for (int i = 0; i < N; i++)
        if (__builtin_amdgcn_ballot_w64(__builtin_isunordered(q[i].x, q[i].y) | __builtin_isunordered(q[i].z, q[i].w)) != 0)
            amax[i] = __builtin_nanf("");
}

// The three INT8 parts of four query elements of a head whose largest magnitude is amax, four codes a
// word. z = q / s_q lies in [-127, 127]; q1 = rint(z), q2 = rint(254 r1) of the remainder r1 = z - q1
// (|r1| <= 1/2) and q3 = rint(254 r2) of r2 = 254 r1 - q2. Adding 1.5 x 2^23 rounds to an integer
// whose low byte is its two's complement code: 7 operations an element where rint, clamp, convert and
// pack took 20 (an instruction of 8 waves on 4 SIMDs: 8 cycles). A NaN leaves code 0: head_max carries it
// into the head's scores.
__device__ __attribute__((always_inline)) inline void query_parts(const float4 &q, float amax, uint32_t (&w)[3]) {
    constexpr float kMagic = 12582912.0f;
    const float inv = amax > 0.0f ? 127.0f / amax : 0.0f;
    const float xs[4] = {q.x, q.y, q.z, q.w};
    uint32_t t[3][4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float t1 = fmaf(xs[e], inv, kMagic), q1 = t1 - kMagic, r1 = fmaf(xs[e], inv, -q1);
        const float t2 = fmaf(r1, 254.0f, kMagic), q2 = t2 - kMagic, r2 = fmaf(r1, 254.0f, -q2);
        const float t3 = fmaf(r2, 254.0f, kMagic);
        t[0][e] = __builtin_bit_cast(uint32_t, t1);
        t[1][e] = __builtin_bit_cast(uint32_t, t2);
        t[2][e] = __builtin_bit_cast(uint32_t, t3);
    }
#pragma unroll
    for (int part = 0; part < 3; part++)
        w[part] = __builtin_amdgcn_perm(t[part][1], t[part][0], 0x0c0c0400u) |
                  __builtin_amdgcn_perm(t[part][3], t[part][2], 0x04000c0cu);
}

// The least reference of a split's V scales: 128 over it is FP32's 2^126. Smaller scales (vectors below
// 1.9e-34) give operands below the full 2^7 instead of an infinite factor.
constexpr float kLeastVScale = 0x1p-119f;

// A split's result is (m, l, O) for l 2^m and O 2^m: O, the sum of up to 2^40 (p <= 2^8, codes and the
// operands' 2^7, 2^18 keys) times the V scale, would pass FP32 where the scale is large, so its factor,
// l's and 2^-m's are then 2^-40 each. (The outputs divide O by l.)
constexpr float kLargeVScale = 0x1p60f;
__device__ inline void shift_large_values(float &vs_out, float &l, float &m) {
    const bool shift = vs_out > kLargeVScale;
    vs_out *= shift ? 0x1p-40f : 1.0f;
    l *= shift ? 0x1p-40f : 1.0f;
    m += shift ? 40.0f : 0.0f;
}

// The exponents' arguments score - ref of a lane's four tokens. One fma of the dot keeps the product
// unrounded, but ref is a rounded score: where scores pass 2^20 the rounding it holds (2^-25 of it) would
// show, and from 2^25 the largest probability no longer fits FP16, or underflows. There the score is
// rounded first, as the one that ref was taken from; per lane, so that a row does not depend on its
// neighbours, and behind `large`, which is wave-uniform and changes with the references only.
__device__ inline bool large_ref(float ref) { return fabsf(ref) > 0x1p20f; }

__device__ __attribute__((always_inline)) inline void exp_args(const float (&dot)[4], float qsc, const float (&ks)[4], float ref,
                                                               bool large, float (&arg)[4]) {
#pragma unroll
    for (int r = 0; r < 4; r++) arg[r] = fmaf(dot[r], qsc * ks[r], -ref);
    if (large) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            float score = dot[r] * (qsc * ks[r]);
            asm("" : "+v"(score));   // (not contracted into an fma again)
            arg[r] = large_ref(ref) ? score - ref : arg[r];
        }
    }
}

// One chunk of one KV group in flight, K and V in separate register sets (K is staged
// one chunk ahead of V): thread t holds K rows t / 16 + 32 i (16 bytes at 16 (t % 16))
// and V page-row segments t / 8 + 64 i (16 bytes at 16 (t % 8)), i < 4: every load
// instruction reads whole 256-byte K rows or whole 128-byte V lines, the pattern that
// streams at full HBM rate (loads shaped like the MFMA operands, 16 rows per
// instruction, reach about two thirds of it).
struct KRegs {
    uint4 k0, k1, k2, k3;   // named, not an array: kept in registers
};
struct VRegs {
    uint4 v0, v1, v2, v3;
};

// The LDS image of a chunk. K: 128 token rows of 256 bytes, 16-byte piece c of
// token t at position c ^ (t % 16). V^T: 256 dimension rows of 128 bytes (the
// chunk's tokens), piece c (tokens 16c..16c+15) of row d at position c ^ ((d / 2) % 8).
// Both make the operand reads and the chunk writes free of bank conflicts.
struct ChunkLds {
    uint4 k[kChunk][16];
    uint4 v[256][8];
};

// The chunk loads are non-temporal (`nt`): each cache byte is read once per step, so it need not
// displace anything in L2 (29.5 instead of 30.6-31.1 us per layer step at 131073).
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

__device__ __attribute__((always_inline)) inline uint4 load_k_piece(const DecodeParams &p, uint32_t g, uint32_t c0,
                                                                    uint32_t length, int tid, int i) {
    const uint32_t t = min(c0 + (uint32_t)(tid >> 4) + 32 * i, length - 1);
    return __builtin_bit_cast(
        uint4, __builtin_nontemporal_load(reinterpret_cast<const u32x4_t *>(p.k + ((size_t)t * 2 + g) * 256 + 16 * (tid & 15))));
}

// 16 bytes as a value (a struct copy straight from global memory would keep the
// register set in a stack object)
__device__ __attribute__((always_inline)) inline uint4 load_piece(const int8_t *at) {
    return __builtin_bit_cast(uint4, __builtin_nontemporal_load(reinterpret_cast<const u32x4_t *>(at)));
}

// K or V of chunk idx of the split starting at token `begin`. Past the last chunk
// (only the prologue's loads of a split shorter than three chunks) the loads stay, a
// fixed count that keeps the counter waits exact, but every lane reads the same 16
// bytes of the first one: a cache line instead of a 32 KB re-read.
__device__ __attribute__((always_inline)) inline void load_k(KRegs &r, const DecodeParams &p, uint32_t g,
                                                             uint32_t begin, uint32_t idx, uint32_t nchunks,
                                                             uint32_t length, int tid) {
    const bool real = idx < nchunks;
    const uint32_t c0 = real ? begin + idx * kChunk : begin;
    const int lt = real ? tid : 0;
    r.k0 = load_k_piece(p, g, c0, length, lt, 0);
    r.k1 = load_k_piece(p, g, c0, length, lt, real ? 1 : 0);
    r.k2 = load_k_piece(p, g, c0, length, lt, real ? 2 : 0);
    r.k3 = load_k_piece(p, g, c0, length, lt, real ? 3 : 0);
}

__device__ __attribute__((always_inline)) inline void load_v(VRegs &r, const DecodeParams &p, uint32_t g,
                                                             uint32_t begin, uint32_t idx, uint32_t nchunks,
                                                             int tid) {
    const bool real = idx < nchunks;
    const uint32_t c0 = real ? begin + idx * kChunk : begin;
    const int lt = real ? tid : 0;
    // c0 is a multiple of 128 inside the cache's whole pages
    const int8_t *vrow = p.v + value_index((uint64_t)c0 * 2 + g, 0) + (size_t)(lt >> 3) * 256 + 16 * (lt & 7);
    const size_t step = real ? 64 * 256 : 0;
    r.v0 = load_piece(vrow);
    r.v1 = load_piece(vrow + step);
    r.v2 = load_piece(vrow + 2 * step);
    r.v3 = load_piece(vrow + 3 * step);
}

__device__ __attribute__((always_inline)) inline void store_k(ChunkLds &b, const KRegs &r, int tid) {
    const int t = tid >> 4, c = tid & 15;   // K rows t + 32i (t + 32i has the same t % 16)
    const int kp = c ^ (t & 15);
    b.k[t][kp] = r.k0;
    b.k[t + 32][kp] = r.k1;
    b.k[t + 64][kp] = r.k2;
    b.k[t + 96][kp] = r.k3;
}

__device__ __attribute__((always_inline)) inline void store_v(ChunkLds &b, const VRegs &r, int tid) {
    const int d = tid >> 3, e = tid & 7;    // V rows d + 64i (same (d / 2) % 8)
    const int vp = e ^ ((d >> 1) & 7);
    b.v[d][vp] = r.v0;
    b.v[d + 64][vp] = r.v1;
    b.v[d + 128][vp] = r.v2;
    b.v[d + 192][vp] = r.v3;
}

// The appended token's bytes in a chunk's registers, just before they are staged: K row `tn` of
// the chunk (held by the 16 threads with tid / 16 == tn % 32, piece tid % 16, in register
// tn / 32) and byte tn % 16 of the 16-token segment tn / 16 of every V page row (threads with
// tid % 8 == tn / 16, rows tid / 8 + 64 i). Whatever the loads returned for that position is
// replaced by the freshly quantized codes.
// (selections are made on 32-bit words with masks: a select between whole uint4 values became a
// select between their addresses and sent the register sets to scratch)
__device__ __attribute__((always_inline)) inline void take_if(uint4 &w, uint32_t keep, const uint4 &f) {
    w.x = (w.x & keep) | (f.x & ~keep);
    w.y = (w.y & keep) | (f.y & ~keep);
    w.z = (w.z & keep) | (f.z & ~keep);
    w.w = (w.w & keep) | (f.w & ~keep);
}

__device__ __attribute__((always_inline)) inline void patch_k(KRegs &r, int tid, int tn, const uint4 *fresh) {
    if ((tid >> 4) != (tn & 31)) return;
    const uint4 f = fresh[tid & 15];
    const int i = tn >> 5;
    take_if(r.k0, i == 0 ? 0u : ~0u, f);
    take_if(r.k1, i == 1 ? 0u : ~0u, f);
    take_if(r.k2, i == 2 ? 0u : ~0u, f);
    take_if(r.k3, i == 3 ? 0u : ~0u, f);
}

__device__ __attribute__((always_inline)) inline uint4 patch_byte(uint4 w, int byte, uint32_t code) {
    const uint32_t sh = 8 * (byte & 3), value = (code & 0xffu) << sh;
    const int word = byte >> 2;
    const uint32_t m0 = word == 0 ? 0xffu << sh : 0u, m1 = word == 1 ? 0xffu << sh : 0u;
    const uint32_t m2 = word == 2 ? 0xffu << sh : 0u, m3 = word == 3 ? 0xffu << sh : 0u;
    w.x = (w.x & ~m0) | (value & m0);
    w.y = (w.y & ~m1) | (value & m1);
    w.z = (w.z & ~m2) | (value & m2);
    w.w = (w.w & ~m3) | (value & m3);
    return w;
}

__device__ __attribute__((always_inline)) inline void patch_v(VRegs &r, int tid, int tn, const uint8_t *fresh) {
    if ((tid & 7) != (tn >> 4)) return;
    const int d = tid >> 3, byte = tn & 15;
    r.v0 = patch_byte(r.v0, byte, fresh[d]);
    r.v1 = patch_byte(r.v1, byte, fresh[d + 64]);
    r.v2 = patch_byte(r.v2, byte, fresh[d + 128]);
    r.v3 = patch_byte(r.v3, byte, fresh[d + 192]);
}

// Grid: (splits, 2 KV groups, rows), one 8-wave work-group per CU; a split is
// split_chunks chunks of 128 tokens, chosen on the host so that the grid fits the
// CUs in one round. The work-group streams its chunks through double-buffered LDS
// with two chunks in flight in registers. Per chunk wave w scores tokens 16w..16w+15,
// S^T[t][n] = K[t] . Qx[n] (16x16x64 INT8 MFMA on the raw K codes, n = 8 heads x
// {q1, q2}, and a second product for q3), and turns them into probabilities in base 2 against a running reference
// shared by the work-group; the waves exchange those P operands through LDS and wave w
// accumulates O^T[d][n] += V^T[d][t] . Px[t][n] for dimensions 32w..32w+31 over all 128
// tokens (16x16x32 FP16 MFMA), so no wave merge of O remains at the end. Px = 2^7 p * vs /
// vs_ref split into FP16 hi + lo; vs_ref, the split's largest V scale, keeps Px below
// 2^15 (p <= 2^8, see below) and vs_ref / 2^7 multiplies the result once. Lane l holds MFMA
// column n = l % 16 and token/k group qq = l / 16.
// Up to about 16000 tokens a split is one chunk and the kernel one chunk's latency, most of it issue
// (an instruction of all eight waves takes 8 cycles of a SIMD): the query's parts are built by a head
// per wave, the prologue has one barrier (two for the work-group that appends), the first chunk's
// operands are made once, after its maxima, and masks are applied only in a row's last chunk. At 777
// tokens 8.9 -> 7.2 us, at 9000 9.4 -> 8.0, at 30000 13.7 -> 12.0; at 131072, where the stream bounds
// it, 28.9 -> 27.2 us (5.0 TB/s).
template <bool kHalfQ>
__global__ __launch_bounds__(512, 1) void decode_int8_kernel(DecodeParams p) {
    typedef int v4i __attribute__((ext_vector_type(4)));
    typedef _Float16 half4 __attribute__((ext_vector_type(4)));
    // the chunk buffers
    __shared__ __attribute__((aligned(16))) unsigned char arena[2 * sizeof(ChunkLds)];
    ChunkLds *bufs = reinterpret_cast<ChunkLds *>(arena);
    __shared__ __attribute__((aligned(16))) float chunk_top[2][16][kDecodeWaves];
    __shared__ float wave_l[kDecodeWaves][16];
    // each wave's P operands, by chunk parity: [wave][column][four of its tokens], as rows_int8_kernel
    __shared__ __attribute__((aligned(16))) uint2 pshare[2][kDecodeWaves][16][4];
    __shared__ __attribute__((aligned(16))) float kscale[kMaxSplitTokens], vscale[kMaxSplitTokens];
    __shared__ float red[kDecodeWaves], qmax[8];
    // append mode: the new token's codes (K row, V column) and scales
    __shared__ __attribute__((aligned(16))) uint8_t fresh_k[256], fresh_v[256];
    __shared__ float fresh_scale[2];
    // INT8 query operands [set][MFMA c][slot] (set 0: q1 | q2 columns, set 1: q3 in columns n < 8),
    // lane (n, qq)'s in slot 16 qq + (n ^ (4 c + qq)) as in rows_int8_kernel, built once and read
    // into registers before the chunk loop. They sit in the V half of chunk buffer 1, which is first
    // written in phase 1, after the barrier that ends phase 0: by then every wave has read its operands.
    v4i(*qlds)[4][64] = reinterpret_cast<v4i(*)[4][64]>(&bufs[1].v[0][0]);
    static_assert(2 * 4 * 64 * sizeof(v4i) <= sizeof(ChunkLds::v), "query operands exceed the V half of a buffer");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = lane & 15, qq = lane >> 4, head = n & 7;
    const bool lo_col = n >= 8;
    const uint32_t split = blockIdx.x, g = blockIdx.y, row = blockIdx.z;
    const uint32_t length = p.pos + row + 1;
    const uint32_t split_tokens = p.split_chunks * kChunk;
    const uint32_t begin = split * split_tokens;
    const uint32_t end = min(length, begin + split_tokens);
    const uint32_t nchunks = end > begin ? (end - begin + kChunk - 1) / kChunk : 0;
    // append mode: the split holding the new token (position pos) stages fresh codes for it
    const bool owner = p.append && begin <= p.pos && p.pos < end;
    const int e_new = owner ? (int)(p.pos - begin) : -1;          // split-local index
    const int jn = owner ? e_new / kChunk : -1, tn = owner ? e_new % kChunk : 0;

    // ---- the small loads first (scales of the split, this wave's query chunk), then
    // the first two chunks: waits on the memory counter are in order, so the set-up
    // below never waits for the chunks
    // (a fixed count of loads, no branches: the counter waits below stay exact;
    // indices past the split repeat its last token, a cache hit)
    uint32_t last = (end > begin ? end : length) - 1;
    if (p.append && last == p.pos && p.pos > 0) last = p.pos - 1;   // its stored scales are stale
    constexpr int kPasses = kMaxSplitTokens / 512;   // (a pass past the split is skipped: uniform)
    float ksv[kPasses], vsv[kPasses];
#pragma unroll
    for (int it = 0; it < kPasses; it++) {
        if (it > 0 && begin + 512 * it >= end) break;
        const size_t at = (size_t)min(begin + tid + 512 * it, last) * 2 + g;
        ksv[it] = p.ks[at];
        vsv[it] = p.vs[at];
    }
    // head `wave` of the group in rope4's layout (dims 4 lane .. +3), and in append mode the new
    // token's K and V of the group (from the query itself when there is no new token: a fixed count
    // of loads keeps the counter waits exact)
    float4 rq;
    if constexpr (kHalfQ) {   // the prefill path's grouped FP16 query, exact in FP32
        const half4 a = *reinterpret_cast<const half4 *>(p.qh + (((size_t)g * p.rows + row) * 8 + wave) * 256 + 4 * lane);
        rq = make_float4((float)a[0], (float)a[1], (float)a[2], (float)a[3]);
    } else {
        rq = *reinterpret_cast<const float4 *>(p.q + ((size_t)row * 16 + g * 8 + wave) * 256 + 4 * lane);
    }
    float4 nk = rq, nv = rq;
    if constexpr (!kHalfQ) {
        const float *knew = p.append ? p.knew : p.q, *vnew = p.append ? p.vnew : p.q;
        nk = *reinterpret_cast<const float4 *>(knew + (size_t)g * 256 + 4 * lane);
        nv = *reinterpret_cast<const float4 *>(vnew + (size_t)g * 256 + 4 * lane);
    }
    // every wave's small loads enter the CU's memory pipeline before any chunk load
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    KRegs ka, kb;   // K of even / odd chunks
    VRegs va, vb;   // V of even / odd chunks
    load_k(ka, p, g, begin, 0, nchunks, length, tid);
    load_v(va, p, g, begin, 0, nchunks, tid);
    load_k(kb, p, g, begin, 1, nchunks, length, tid);
    load_v(vb, p, g, begin, 1, nchunks, tid);

    float vmax[1] = {0.0f};
    if (p.append) {
        // the same rotation (and, for the new token, quantization) as batch_rope_int8
        // (kv_store.hip), so the cache bytes and the rotated query match it bit for bit
        const float ifreq = lane_inv_freq(p.freq);
        const Rope4 r = rope_angles(p.pos, lane, ifreq);
        rq = rope4(rq, lane, r);
        if (owner) {
            *reinterpret_cast<float4 *>(p.rotated + ((size_t)g * 8 + wave) * 256 + 4 * lane) = rq;
            const uint64_t vector = (uint64_t)p.pos * 2 + g;
            if (wave == 0) {
                const float4 kz = rope4(nk, lane, r);
                const float ka = wave_max(fmaxf(fmaxf(fabsf(kz.x), fabsf(kz.y)), fmaxf(fabsf(kz.z), fabsf(kz.w))));
                const float kr127 = 127.0f / ka;
                const uint32_t codes = pack4(quant_code(kz.x, ka, kr127), quant_code(kz.y, ka, kr127),
                                             quant_code(kz.z, ka, kr127), quant_code(kz.w, ka, kr127));
                *reinterpret_cast<uint32_t *>(p.k_out + vector * 256 + 4 * lane) = codes;
                *reinterpret_cast<uint32_t *>(&fresh_k[4 * lane]) = codes;
                if (lane == 0) {
                    p.ks_out[vector] = ka / 127.0f;
                    fresh_scale[0] = ka / 127.0f;
                }
            } else if (wave == 1) {
                const float va = wave_max(fmaxf(fmaxf(fabsf(nv.x), fabsf(nv.y)), fmaxf(fabsf(nv.z), fabsf(nv.w))));
                const float vr127 = 127.0f / va;
                const float c[4] = {quant_code(nv.x, va, vr127), quant_code(nv.y, va, vr127),
                                    quant_code(nv.z, va, vr127), quant_code(nv.w, va, vr127)};
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint8_t b = (uint8_t)(int8_t)(int)c[i];
                    p.v_out[value_index(vector, 4 * lane + i)] = (int8_t)b;
                    fresh_v[4 * lane + i] = b;
                }
                if (lane == 0) {
                    p.vs_out[vector] = va / 127.0f;
                    fresh_scale[1] = va / 127.0f;
                }
            }
            __syncthreads();   // the fresh codes and scales are in LDS (owner is work-group-uniform)
        }
    }
    // ---- the INT8 parts of head `wave`, one lane's four dimensions (as rows_int8_kernel: each wave
    // one head, where every wave built a quarter of all eight and the maxima met behind a barrier)
    {
        const float4 x[1] = {rq};
        float amax[1];
        head_max(x, amax);
        uint32_t w[3];
        query_parts(rq, amax[0], w);
        const int c = lane >> 4, bq = (lane >> 2) & 3, mix = 4 * c + bq;
        reinterpret_cast<uint32_t *>(&qlds[0][c][16 * bq + (wave ^ mix)])[lane & 3] = w[0];
        reinterpret_cast<uint32_t *>(&qlds[0][c][16 * bq + ((8 + wave) ^ mix)])[lane & 3] = w[1];
        reinterpret_cast<uint32_t *>(&qlds[1][c][16 * bq + (wave ^ mix)])[lane & 3] = w[2];
        if (lane == 0) qmax[wave] = amax[0];
    }
    // ---- the split's scales (this group) into LDS, vs_ref = the maximum of its V scales; entries past
    // the split are zero, the new token's from its fresh scales
#pragma unroll
    for (int it = 0; it < kPasses; it++) {
        if (it > 0 && begin + 512 * it >= end) break;
        const uint32_t e = tid + 512 * it;
        const bool inside = begin + e < end, fresh = (int)e == e_new;
        const float sk = fresh ? fresh_scale[0] : ksv[it], sv = fresh ? fresh_scale[1] : vsv[it];
        kscale[e] = inside ? sk * (kLog2e / 16.0f / 254.0f) : 0.0f;   // a dot's unit is 1 / 254 (below)
        vscale[e] = inside ? sv : 0.0f;
        vmax[0] = fmaxf(vmax[0], inside ? sv : 0.0f);
    }
    wave_allmax(vmax);
    if (lane == 0) red[wave] = vmax[0];
    // K of chunk 0 into buffer 0 and K of chunk 2 into the registers it leaves
    if (jn == 0) patch_k(ka, tid, tn, reinterpret_cast<const uint4 *>(fresh_k));
    store_k(bufs[0], ka, tid);
    load_k(ka, p, g, begin, 2, nchunks, length, tid);
    __syncthreads();
    float vs_ref = red[0];
#pragma unroll
    for (int w = 1; w < kDecodeWaves; w++) vs_ref = fmaxf(vs_ref, red[w]);
    // operands up to 2^8 times 2^7 stay below FP16's 65504; the factor keeps their lo parts out of its
    // subnormals
    vs_ref = fmaxf(vs_ref, kLeastVScale);
    const float vs_inv = 128.0f / vs_ref;
    vs_ref *= 1.0f / 128.0f;
    const float qsc = qmax[head] * (1.0f / 127.0f);   // s_q of the lane's head
    v4i qi[4], q3i[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        qi[c] = qlds[0][c][16 * qq + (n ^ (4 * c + qq))];
        q3i[c] = qlds[1][c][16 * qq + (head ^ (4 * c + qq))];
    }

    floatx4 o[2];   // O^T tiles dt = 2 wave + i, over every token of the split
    o[0] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    o[1] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    float m = -INFINITY, l = 0.0f, total_prev = 0.0f;   // l: this lane's tokens, summed at the end
    float dot_prev[4] = {0.0f, 0.0f, 0.0f, 0.0f};   // the previous chunk's dots, for a rebuild of its operands
    bool large = false;   // some column's reference is large (exp_args)

    // Probabilities of the lane's four tokens of chunk j against the running reference, as the FP16 hi
    // (column n < 8) or lo (n >= 8) part of p * vs / vs_ref, published as this wave's P operand;
    // total_prev = the lane's sum.
    auto probs = [&](uint32_t j) __attribute__((always_inline)) {
        const int local0 = (int)(j * kChunk) + 16 * wave + 4 * qq;   // token offset inside the split
        const float4 vs4 = *reinterpret_cast<const float4 *>(&vscale[local0]);
        const float4 ks4 = *reinterpret_cast<const float4 *>(&kscale[local0]);
        const float vsr[4] = {vs4.x, vs4.y, vs4.z, vs4.w}, ksr[4] = {ks4.x, ks4.y, ks4.z, ks4.w};
        const float refc = fmaxf(m, -3.0e38f);   // m = -inf only in a column without a score yet
        float arg[4];
        exp_args(dot_prev, qsc, ksr, refc, large, arg);
        if (begin + (j + 1) * kChunk > end)   // uniform: only a row's last chunk holds tokens past its end
#pragma unroll
            for (int r = 0; r < 4; r++) arg[r] = begin + local0 + r < end ? arg[r] : -INFINITY;
        half4 pop;
        total_prev = 0.0f;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float prob = __builtin_amdgcn_exp2f(arg[r]);   // 0 for masked tokens
            total_prev += prob;
            float scaled = prob * (vsr[r] * vs_inv);
            asm("" : "+v"(scaled));   // one rounded value for both parts (see rows_int8_kernel)
            const _Float16 hi = (_Float16)scaled;
            pop[r] = lo_col ? (_Float16)(scaled - (float)hi) : hi;
        }
        pshare[j & 1][wave][n][qq] = __builtin_bit_cast(uint2, pop);
    };
    // Phase j (one barrier each): finish chunk j - 1 (the rescale decision, then PV), score
    // chunk j, store V of chunk j and K of chunk j + 1, load V of chunk j + 2 and K of chunk
    // j + 3 into the registers just stored. K is staged one chunk ahead of V, so the two
    // buffers' K and V halves have different lifetimes: in phase j chunk j - 1's V and chunk
    // j's K are read while chunk j's V and chunk j + 1's K are written.
    // The waves share one running reference m per column; a chunk rescales (and pays a
    // second barrier) only when some column's maximum passes m by more than 2^8, so
    // p = 2^(s - m) stays below 256.
    auto finish = [&](uint32_t j) __attribute__((always_inline)) {   // chunk j - 1, j > 0
        {
            const int slot = (j - 1) & 1;
            const float4 ta = *reinterpret_cast<const float4 *>(&chunk_top[slot][n][0]);
            const float4 tb = *reinterpret_cast<const float4 *>(&chunk_top[slot][n][4]);
            const float ctop = fmaxf(fmaxf(fmaxf(ta.x, ta.y), fmaxf(ta.z, ta.w)), fmaxf(fmaxf(tb.x, tb.y), fmaxf(tb.z, tb.w)));
            // every wave reads the same maxima: the branch is uniform over the work-group. Chunk 0 has
            // no reference before its maxima: its operands are made here
            if (j == 1 || __builtin_amdgcn_ballot_w64(ctop > m + 8.0f) != 0) {
                const float next = fmaxf(m, ctop);
                const float decay = next == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - next);
                l *= decay;
                o[0] *= decay;
                o[1] *= decay;
                m = next;
                large = __builtin_amdgcn_ballot_w64(large_ref(m)) != 0;
                probs(j - 1);   // no wave reads the slot before this branch
                __syncthreads();
            }
            l += total_prev;
            // O^T[d][n] += V^T[d][t] P[t][n] for this wave's 32 dimensions over the chunk's 128
            // tokens on v_mfma_f32_16x16x32_f16: k-step s takes waves 2s and 2s + 1's tokens (32),
            // lane (n, qq) tokens 8 (qq % 2) .. + 7 of wave 2s + qq / 2, i.e. the published P
            // operands 2 (qq % 2) and 2 (qq % 2) + 1 of column n and 8 codes
            // (one 8-byte read) of its V piece. Against 16 MFMAs of 16 tokens with a 4-byte read
            // each: half the MFMAs, dependent steps and V reads (29.6-30.0 against 30.2-30.3 us
            // per layer step at 131073)
            const ChunkLds &b = bufs[slot];
#pragma unroll
            for (int s = 0; s < kDecodeWaves / 2; s++) {
                const int src = 2 * s + (qq >> 1);
                const half8 ps = *reinterpret_cast<const half8 *>(&pshare[slot][src][n][2 * (qq & 1)]);
#pragma unroll
                for (int jj = 0; jj < 2; jj++) {
                    const int d = 16 * (2 * wave + jj) + n;
                    const uint2 w8 = reinterpret_cast<const uint2 *>(&b.v[d][src ^ ((d >> 1) & 7)])[qq & 1];
                    uint32_t h0, h1, h2, h3;
                    i8x8_to_f16_sdwa(w8.x, w8.y, h0, h1, h2, h3);
                    const half8 va8 = __builtin_bit_cast(half8, make_uint4(h0, h1, h2, h3));
                    o[jj] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va8, ps, o[jj], 0, 0, 0);
                }
            }
        }
    };
    // odd: a compile-time parity of j, which picks the register sets (V of chunk j, K of
    // chunk j + 1) without taking their addresses
    auto phase = [&](uint32_t j, auto odd, bool store_knext, bool load_v2, bool load_k3) __attribute__((always_inline)) {
        VRegs &rv = decltype(odd)::value ? vb : va;
        KRegs &rk = decltype(odd)::value ? ka : kb;
        if (j > 0) finish(j);
        {
            const ChunkLds &b = bufs[j & 1];
            const int tl = 16 * wave + (lane & 15);          // the lane's K row of the chunk
            // S^T: rows = tokens 16w + 4qq + r of the chunk, columns n; acc3 holds the q3 part
            v4i acc = {0, 0, 0, 0}, acc3 = {0, 0, 0, 0};
#pragma unroll
            for (int jj = 0; jj < 4; jj++) {
                const v4i kop = __builtin_bit_cast(v4i, b.k[tl][(4 * jj + qq) ^ (tl & 15)]);
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(kop, qi[jj], acc, 0, 0, 0);
                acc3 = __builtin_amdgcn_mfma_i32_16x16x64_i8(kop, q3i[jj], acc3, 0, 0, 0);
            }
            // column n holds the q1 dots (n < 8) or the q2 dots of head n % 8, and the partner column
            // the other: 254 dot1 + dot2 is an exact integer (|dots| < 2^22), summed over the pair by
            // one DPP add. The exponent's argument is one fma of the dot (probs), so the score itself,
            // rounded, is only compared
            const int local0 = (int)(j * kChunk) + 16 * wave + 4 * qq;   // token offset inside the split
            const float4 ks4 = *reinterpret_cast<const float4 *>(&kscale[local0]);
            const float ksr[4] = {ks4.x, ks4.y, ks4.z, ks4.w};
            float score[4];
            int d12[4];
#pragma unroll
            for (int r = 0; r < 4; r++) d12[r] = __mul24(acc[r], lo_col ? 1 : 254);
            add_row_partner8(d12);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                dot_prev[r] = fmaf((float)acc3[r], 1.0f / 254.0f, (float)d12[r]);
                score[r] = dot_prev[r] * (qsc * ksr[r]);
            }
            if (begin + (j + 1) * kChunk > end)
#pragma unroll
                for (int r = 0; r < 4; r++) score[r] = begin + local0 + r < end ? score[r] : -INFINITY;
            const float top = xl_max32(xl_max16(fmaxf(fmaxf(score[0], score[1]), fmaxf(score[2], score[3]))));
            if (qq == 0) chunk_top[j & 1][n][wave] = top;
            if (j > 0) probs(j);
        }
        if ((int)j == jn) patch_v(rv, tid, tn, fresh_v);
        store_v(bufs[j & 1], rv, tid);
        if (load_v2) load_v(rv, p, g, begin, j + 2, nchunks, tid);
        if ((int)j + 1 == jn) patch_k(rk, tid, tn, reinterpret_cast<const uint4 *>(fresh_k));
        if (store_knext) store_k(bufs[(j + 1) & 1], rk, tid);
        if (load_k3) load_k(rk, p, g, begin, j + 3, nchunks, length, tid);
        __syncthreads();
    };
    // Phases in pairs, so that the register sets keep fixed roles without copies (a copy of
    // registers still being loaded waits for the load). The pairs run while every load is
    // a real chunk (a fixed count per pair keeps the counter waits exact); the last one to
    // four chunks follow without loads past the end, whose registers the end of the
    // work-group would otherwise wait for.
    uint32_t c = 0;
    for (; c + 4 < nchunks; c += 2) {
        phase(c, std::false_type{}, true, true, true);
        phase(c + 1, std::true_type{}, true, true, true);
    }
    if (c < nchunks) {
        phase(c, std::false_type{}, c + 1 < nchunks, c + 2 < nchunks, c + 3 < nchunks);
        uint32_t last_phase = c + 1;
        if (c + 1 < nchunks) {
            phase(c + 1, std::true_type{}, c + 2 < nchunks, c + 3 < nchunks, false);
            last_phase = c + 2;
            if (c + 2 < nchunks) {
                phase(c + 2, std::false_type{}, c + 3 < nchunks, false, false);
                last_phase = c + 3;
                if (c + 3 < nchunks) {
                    phase(c + 3, std::true_type{}, false, false, false);
                    last_phase = c + 4;
                }
            }
        }
        finish(last_phase);
    }

    // ---- the waves share m; l sums over waves. O^T[d][n], d = 16 dt + 4 qq + r: the lo
    // column n + 8 of each head joins its hi column n in registers (the DPP adds take MFMA
    // results as inline-assembly operands, for which the compiler inserts no wait states:
    // cover them here), then lanes n < 8 hold tile 2 wave and lanes n >= 8 tile 2 wave + 1.
    l = xl_sum32(xl_sum16(l));
    shift_large_values(vs_ref, l, m);
    if (qq == 0) wave_l[wave][n] = l;
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7");
    __builtin_amdgcn_sched_barrier(0);
    add_row_partner8(o[0], o[1]);
    const bool upper = n >= 8;
    const int d0 = 16 * (2 * wave + (upper ? 1 : 0)) + 4 * qq;
    const int h = head;
    floatx4 res = upper ? o[1] : o[0];
    float4 acc = make_float4(res[0] * vs_ref, res[1] * vs_ref, res[2] * vs_ref, res[3] * vs_ref);
    if (p.splits == 1) {
        // gate and y need only 4-byte alignment
        // (the four gate loads go out before the first store: the compiler cannot tell y from gate)
        const size_t at = ((size_t)row * 16 + g * 8 + h) * 256 + d0;
        const float g0 = p.gate[at + 0], g1 = p.gate[at + 1], g2 = p.gate[at + 2], g3 = p.gate[at + 3];
        asm volatile("" ::"v"(g0), "v"(g1), "v"(g2), "v"(g3) : "memory");
        __syncthreads();
        float lw = 0.0f;
#pragma unroll
        for (int w = 0; w < kDecodeWaves; w++) lw += wave_l[w][head];
        const float inv = 1.0f / lw;
        p.y[at + 0] = acc.x * inv * sigmoidf(g0);
        p.y[at + 1] = acc.y * inv * sigmoidf(g1);
        p.y[at + 2] = acc.z * inv * sigmoidf(g2);
        p.y[at + 3] = acc.w * inv * sigmoidf(g3);
        return;
    }
    float *part = p.partial + (((size_t)row * 2 + g) * p.splits + split) * kPartialFloats;
    *reinterpret_cast<float4 *>(part + h * 256 + d0) = acc;   // needs no other wave's l
    __syncthreads();
    if (wave == 0 && lane < 8) {
        float lw = 0.0f;
#pragma unroll
        for (int w = 0; w < kDecodeWaves; w++) lw += wave_l[w][head];
        part[2048 + h] = m;
        part[2056 + h] = lw;
    }
}

// Merges the splits of one (row, head) (grid: 4 x 16 heads x rows, four waves per work-group).
// Each wave owns 16 dimensions and works alone (no LDS, no barrier): lane (sg, q) holds the
// float4 of dimensions 4q .. 4q + 3 for splits sg, sg + 16, ... (the first 128 splits' m, l and
// partials loaded at once), the maximum of m and then the weighted sums of l and O are reduced
// over the 16 split groups, and the lanes of group 0 write the output. The order of every sum
// is fixed by the split count alone.
__global__ __launch_bounds__(256) void decode_combine_kernel(const float *__restrict__ partial, const float *__restrict__ gate,
                                                             float *__restrict__ y, uint32_t splits) {
    const uint32_t row = blockIdx.z, hq = blockIdx.y, g = hq / 8, h = hq % 8;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int q = lane & 3, sg = lane >> 2;
    const uint32_t d = (blockIdx.x * 4 + wave) * 16 + 4 * q;
    const float *base = partial + ((size_t)row * 2 + g) * splits * kPartialFloats;
    constexpr int kEarly = 8;
    float mv[kEarly], lv[kEarly];
    float4 ov[kEarly];
#pragma unroll
    for (int u = 0; u < kEarly; u++) {
        const uint32_t s = sg + 16 * u, sidx = min(s, splits - 1);
        const float *sp = base + (size_t)sidx * kPartialFloats;
        ov[u] = *reinterpret_cast<const float4 *>(sp + h * 256 + d);
        mv[u] = s < splits ? sp[2048 + h] : -INFINITY;
        lv[u] = sp[2056 + h];
    }
    const size_t at = ((size_t)row * 16 + hq) * 256 + d;
    float gv[4];
#pragma unroll
    for (int i = 0; i < 4; i++) gv[i] = gate[at + i];   // y and gate need only 4-byte alignment
    float mmax = mv[0];
#pragma unroll
    for (int u = 1; u < kEarly; u++) mmax = fmaxf(mmax, mv[u]);
    for (uint32_t s = sg + 16 * kEarly; s < splits; s += 16) mmax = fmaxf(mmax, base[(size_t)s * kPartialFloats + 2048 + h]);
#pragma unroll
    for (int o = 4; o < 64; o <<= 1) mmax = fmaxf(mmax, __shfl_xor(mmax, o, 64));
    float lsum = 0.0f;
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    auto add = [&](float m, float l, const float4 &o) {
        if (m == -INFINITY) return;   // a split that holds none of the row's keys
        const float w = __builtin_amdgcn_exp2f(m - mmax);
        lsum += l * w;
        acc.x += o.x * w;
        acc.y += o.y * w;
        acc.z += o.z * w;
        acc.w += o.w * w;
    };
#pragma unroll
    for (int u = 0; u < kEarly; u++) add(mv[u], lv[u], ov[u]);
    for (uint32_t s = sg + 16 * kEarly; s < splits; s += 16) {
        const float *sp = base + (size_t)s * kPartialFloats;
        add(sp[2048 + h], sp[2056 + h], *reinterpret_cast<const float4 *>(sp + h * 256 + d));
    }
#pragma unroll
    for (int o = 4; o < 64; o <<= 1) {
        lsum += __shfl_xor(lsum, o, 64);
        acc.x += __shfl_xor(acc.x, o, 64);
        acc.y += __shfl_xor(acc.y, o, 64);
        acc.z += __shfl_xor(acc.z, o, 64);
        acc.w += __shfl_xor(acc.w, o, 64);
    }
    if (sg == 0) {
        const float inv = 1.0f / lsum;
        y[at + 0] = acc.x * inv * sigmoidf(gv[0]);
        y[at + 1] = acc.y * inv * sigmoidf(gv[1]);
        y[at + 2] = acc.z * inv * sigmoidf(gv[2]);
        y[at + 3] = acc.w * inv * sigmoidf(gv[3]);
    }
}

// ---------------------------------------------------------------- several rows per work-group

// Attention of up to 2 CT rows against one staging of the keys: verify blocks (FP32 query) and
// prefill chunks over short key ranges (grouped FP16 query). The
// decode kernel above gives each row a work-group of its own, so R rows read, stage and convert
// the cache R times, and the three-kernel reader (five launches) writes every score to memory and
// reads it back twice. Per layer, with the combine, against the reader: 8 rows after 1500 keys 12.8
// (40.0) us, where either is launches and one chunk's latency; 4 rows after 30000 keys 21.9 (47.6)
// us, 1.4 TB/s of cache: bound by the issue of a chunk's vector and matrix work and the start of a
// work-group, not by the stream.
//
// Grid: (split, KV group) pairs x row blocks, one 8-wave work-group per CU; the row blocks of a pair
// are 8 blocks apart, on one XCD, whose L2 serves the second and later ones. A split is split_chunks
// chunks of 128 tokens, streamed as in decode_int8_kernel, with the same arithmetic (three INT8
// query parts, FP16 hi + lo probabilities, lazy running maxima), and these differences:
//   * 16 MFMA columns are two rows x 8 heads, for each of q1, q2, q3 (the three parts of a score meet
//     in one lane) and for P's hi and lo parts (which accumulate into one O), so no column computes
//     another's exponentials and nothing is exchanged between column halves;
//   * wave w stages its own 16 K rows in an LDS slice that no other wave reads (whole 256-byte rows
//     per load, no barrier); V and P are shared as there;
//   * every quantity of a column (its running maximum and rescales, its V scale reference over the
//     tokens it sees) depends on that row alone, and split boundaries are absolute, so a row's result
//     does not depend on the rows dispatched with it: a verify block's rows are bitwise those of any
//     shorter block or slice.
// 4 rows keep two of their three query parts in 64 registers, the third in LDS; 8 rows would need
// twice that, and 64 KB of LDS for their P operands beside the 112 KB of staging and scales.
struct RowsParams {
    const float *q;         // FP32 [rows][16][256], or
    const _Float16 *qh;     // kHalfQ: the grouped FP16 query [2][rows][8][256]
    const int8_t *k;
    const int8_t *v;
    const float *ks;
    const float *vs;
    const float *gate;
    float *y;
    float *partial;   // as decode_int8_kernel's
    uint32_t rows, pos, splits, split_chunks, zs;   // zs: row blocks
};

template <int CT, bool kOnce, bool kHalfQ>
__global__ __launch_bounds__(512, 1) void rows_int8_kernel(RowsParams p) {
    typedef int v4i __attribute__((ext_vector_type(4)));
    typedef _Float16 half4 __attribute__((ext_vector_type(4)));
    constexpr int kRowsPer = 2 * CT;
    __shared__ uint4 vbuf[2][256][8];                        // V chunks by parity, as ChunkLds::v
    __shared__ uint4 kbuf[kDecodeWaves][16][16];             // each wave's K rows, piece c of row t at c ^ t
    // P operands [parity][tile][hi, lo][wave][column][four of the wave's tokens]: a PV step's eight
    // tokens are one 16-byte read, a wave's reads and writes contiguous
    __shared__ __attribute__((aligned(16))) uint2 pshare[2][CT][2][kDecodeWaves][16][4];
    __shared__ __attribute__((aligned(16))) float kscale[kMaxSplitTokens], vscale[kMaxSplitTokens];
    __shared__ __attribute__((aligned(16))) float chunk_top[2][CT][16][kDecodeWaves];
    __shared__ float wave_l[CT][kDecodeWaves][16];
    __shared__ float red[kDecodeWaves], qmax[CT][16];
    // the query operands [tile][part][64-dimension step c][slot], lane (n, qq)'s in slot
    // 16 qq + (n ^ (4 c + qq)), so that the 4-byte writes below spread over the banks: q1 and q2, built once and read into
    // registers, in V buffer 1, which is first written in phase 1, after the barrier that ends phase 0;
    // q3 stays in LDS (in registers it spilled, and a reload waits for the chunk loads before it)
    v4i(*qlds)[2][4][64] = reinterpret_cast<v4i(*)[2][4][64]>(&vbuf[1][0][0]);
    static_assert(CT * 2 * 4 * 64 * sizeof(v4i) <= sizeof(vbuf[0]), "query operands exceed a V buffer");
    __shared__ v4i q3lds[CT][4][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = lane & 15, qq = lane >> 4, head = n & 7;
    uint32_t pair, zb;
    if constexpr (kHalfQ) {   // pairs in turn: few pairs and many row blocks must reach every XCD
        pair = blockIdx.x % (2 * p.splits);
        zb = blockIdx.x / (2 * p.splits);
    } else {
        const uint32_t jb = blockIdx.x / 8;
        pair = (jb / p.zs) * 8 + blockIdx.x % 8;
        zb = jb % p.zs;
        if (pair >= 2 * p.splits) return;   // padding of the grid to whole rounds of 8
    }
    const uint32_t split = pair >> 1, g = pair & 1, r0 = zb * kRowsPer;
    const uint32_t nr = min((uint32_t)kRowsPer, p.rows - r0);
    const uint32_t first_end = p.pos + r0 + 1, block_end = p.pos + r0 + nr;   // keys of the first and last row
    const uint32_t begin = split * p.split_chunks * kChunk;
    const uint32_t end = min(block_end, begin + p.split_chunks * kChunk);
    auto part_of = [&](uint32_t ri) __attribute__((always_inline)) {
        return p.partial + (((size_t)(r0 + ri) * 2 + g) * p.splits + split) * kPartialFloats;
    };
    if (begin >= block_end) {   // no keys of these rows (only with several splits): an empty partial
        if (tid < 8 * (int)nr) part_of(tid >> 3)[2048 + (tid & 7)] = -INFINITY;
        return;
    }
    const uint32_t nchunks = (end - begin + kChunk - 1) / kChunk;

    // ---- the small loads first, then the first chunk (as decode_int8_kernel)
    const uint32_t last = end - 1;
    // (the scales of a split of up to 512 tokens in one load each: the counts of further passes are
    // uniform branches)
    constexpr int kPasses = kMaxSplitTokens / 512;
    float ksv[kPasses], vsv[kPasses], vnew[kRowsPer];
#pragma unroll
    for (int it = 0; it < kPasses; it++) {
        if (it > 0 && begin + 512 * it >= end) break;
        const size_t at = (size_t)min(begin + tid + 512 * it, last) * 2 + g;
        ksv[it] = p.ks[at];
        vsv[it] = p.vs[at];
    }
    // the V scales of the tokens between the first and the last row's ends
#pragma unroll
    for (int i = 0; i + 1 < kRowsPer; i++) vnew[i] = p.vs[(size_t)min(first_end + i, last) * 2 + g];
    // wave w builds the operands of head w of every row, lane holding dimensions 4 lane .. + 3
    float4 x[kRowsPer];
#pragma unroll
    for (int r = 0; r < kRowsPer; r++) {
        const uint32_t row = r0 + min((uint32_t)r, nr - 1);
        if constexpr (kHalfQ) {   // exact in FP32
            const half4 a = *reinterpret_cast<const half4 *>(p.qh + (((size_t)g * p.rows + row) * 8 + wave) * 256 + 4 * lane);
            x[r] = make_float4((float)a[0], (float)a[1], (float)a[2], (float)a[3]);
        } else {
            x[r] = *reinterpret_cast<const float4 *>(p.q + ((size_t)row * 16 + g * 8 + wave) * 256 + 4 * lane);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    // kOnce: the codes are read by this work-group only (one row block) and need not stay in L2
    auto load16 = [&](const int8_t *at) __attribute__((always_inline)) {
        if constexpr (kOnce) return load_piece(at);
        return *reinterpret_cast<const uint4 *>(at);
    };
    // K rows 16 wave + 4 i + lane / 16 of chunk idx, piece lane % 16; V segments as decode_int8_kernel's
    auto load_k = [&](KRegs &r, uint32_t idx) __attribute__((always_inline)) {
        const uint32_t t = begin + idx * kChunk + 16 * wave + (lane >> 4);
        const int8_t *base = p.k + (size_t)g * 256 + 16 * (lane & 15);
        r.k0 = load16(base + (size_t)min(t, last) * 512);
        r.k1 = load16(base + (size_t)min(t + 4, last) * 512);
        r.k2 = load16(base + (size_t)min(t + 8, last) * 512);
        r.k3 = load16(base + (size_t)min(t + 12, last) * 512);
    };
    auto load_v = [&](VRegs &r, uint32_t idx) __attribute__((always_inline)) {
        const int8_t *vrow = p.v + value_index((uint64_t)(begin + idx * kChunk) * 2 + g, 0) + (size_t)(tid >> 3) * 256 + 16 * (tid & 7);
        r.v0 = load16(vrow);
        r.v1 = load16(vrow + 64 * 256);
        r.v2 = load16(vrow + 128 * 256);
        r.v3 = load16(vrow + 192 * 256);
    };
    auto store_k = [&](const KRegs &r) __attribute__((always_inline)) {
        const int t = lane >> 4, c = lane & 15;
        kbuf[wave][t][c ^ t] = r.k0;
        kbuf[wave][t + 4][c ^ (t + 4)] = r.k1;
        kbuf[wave][t + 8][c ^ (t + 8)] = r.k2;
        kbuf[wave][t + 12][c ^ (t + 12)] = r.k3;
    };
    auto store_v = [&](int slot, const VRegs &r) __attribute__((always_inline)) {
        const int d = tid >> 3, vp = (tid & 7) ^ ((d >> 1) & 7);   // V rows d + 64 i (same (d / 2) % 8)
        vbuf[slot][d][vp] = r.v0;
        vbuf[slot][d + 64][vp] = r.v1;
        vbuf[slot][d + 128][vp] = r.v2;
        vbuf[slot][d + 192][vp] = r.v3;
    };
    // One register set each for K and V: a chunk's loads have a whole phase (about 2 us) to arrive. A
    // second set, 32 registers that the operand reads then run ahead in, measured slower: 4 rows after
    // 1500 keys 9.5 against 8.5 us, after 30000 19.1 against 17.6, 1 row after 100000 22.7 against 20.9.
    KRegs rk;
    VRegs rv;
    load_k(rk, 0);
    load_v(rv, 0);

    // ---- the query's INT8 parts
    float amax[kRowsPer];
    head_max(x, amax);
#pragma unroll
    for (int r = 0; r < kRowsPer; r++) {
        uint32_t w[3];
        query_parts(x[r], amax[r], w);
        // dimension 4 lane: step c, block bq (of the operand's lanes), word lane % 4 of its 16 bytes
        const int c = lane >> 4, bq = (lane >> 2) & 3, col = 8 * (r & 1) + wave;
        const int slot = 16 * bq + (col ^ (4 * c + bq));
        reinterpret_cast<uint32_t *>(&qlds[r >> 1][0][c][slot])[lane & 3] = w[0];
        reinterpret_cast<uint32_t *>(&qlds[r >> 1][1][c][slot])[lane & 3] = w[1];
        reinterpret_cast<uint32_t *>(&q3lds[r >> 1][c][slot])[lane & 3] = w[2];
        if (lane == 0) qmax[r >> 1][col] = amax[r];
    }
    // ---- scales of the split into LDS, the work-group's largest V scale
    float vmax[1] = {0.0f};
#pragma unroll
    for (int it = 0; it < kPasses; it++) {
        if (it > 0 && begin + 512 * it >= end) break;
        const uint32_t e = tid + 512 * it, t = begin + e;
        kscale[e] = t < end ? ksv[it] * (kLog2e / 16.0f / 254.0f) : 0.0f;   // a dot's unit is 1 / 254 (below)
        vscale[e] = t < end ? vsv[it] : 0.0f;
        vmax[0] = fmaxf(vmax[0], t < min(end, first_end) ? vsv[it] : 0.0f);
    }
    wave_allmax(vmax);
    if (lane == 0) red[wave] = vmax[0];
    store_k(rk);
    if (1 < nchunks) load_k(rk, 1);
    __syncthreads();
    // row i of the block sees the tokens before first_end and vnew[0 .. i - 1], where the split holds them
    float vcum = red[0];
#pragma unroll
    for (int w = 1; w < kDecodeWaves; w++) vcum = fmaxf(vcum, red[w]);
    float vref[CT], vinv[CT], qsc[CT];
    uint32_t row_end[CT];   // keys the column's row sees (a missing row repeats the last one)
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
        float two[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int ri = 2 * ct + i;
            if (ri > 0) {
                const uint32_t t = first_end + ri - 1;
                vcum = fmaxf(vcum, t >= begin && t < end ? vnew[ri - 1] : 0.0f);
            }
            two[i] = vcum;
        }
        const float even = two[0], odd = two[1];
        vref[ct] = n >= 8 ? odd : even;
        // operands up to 2^8 times 2^7 stay below FP16's 65504; the factor keeps their lo parts out of
        // its subnormals
        vref[ct] = fmaxf(vref[ct], kLeastVScale);
        vinv[ct] = 128.0f / vref[ct];
        vref[ct] *= 1.0f / 128.0f;
        qsc[ct] = qmax[ct][n] * (1.0f / 127.0f);
        row_end[ct] = first_end + min((uint32_t)(2 * ct + (n >> 3)), nr - 1);
    }
    v4i qi[CT][2][4];
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
#pragma unroll
        for (int part = 0; part < 2; part++)
#pragma unroll
            for (int c = 0; c < 4; c++) qi[ct][part][c] = qlds[ct][part][c][16 * qq + (n ^ (4 * c + qq))];

    // O^T of the wave's 32 dimensions. A prefill chunk holds it as one 32x32 tile, element e of a lane
    // being dimension 32 wave + 8 (e / 4) + 4 (lane / 32) + e % 4 of column lane % 32 (tile oct, column
    // n); verify rows, which must come out the same in one tile and in two, as 16x16 tiles
    constexpr bool kWide = kHalfQ;
    static_assert(!kWide || CT == 2, "a 32x32 tile holds two tiles' columns");
    const int oct = (lane >> 4) & 1;
    floatx16 ow;
    floatx4 o[2][CT];   // 16x16: dimensions 32 wave + 16 dt + 4 qq + r of column n
    float m[CT], l[CT], total_prev[CT], dot_prev[CT][4];   // l: this lane's tokens, summed over lanes at the end
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
        o[0][ct] = o[1][ct] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        m[ct] = -INFINITY;
        l[ct] = total_prev[ct] = 0.0f;
#pragma unroll
        for (int r = 0; r < 4; r++) dot_prev[ct][r] = 0.0f;
    }
    bool large = false;   // some column's reference is large (exp_args)
    auto probs = [&](uint32_t j) __attribute__((always_inline)) {
        const int slot = j & 1, local0 = (int)(j * kChunk) + 16 * wave + 4 * qq;
        const float4 vs4 = *reinterpret_cast<const float4 *>(&vscale[local0]);
        const float4 ks4 = *reinterpret_cast<const float4 *>(&kscale[local0]);
        const float vsr[4] = {vs4.x, vs4.y, vs4.z, vs4.w}, ksr[4] = {ks4.x, ks4.y, ks4.z, ks4.w};
        const uint32_t t0 = begin + (uint32_t)local0;
        const bool edge = begin + (j + 1) * kChunk > first_end;   // some row does not see the whole chunk
#pragma unroll
        for (int ct = 0; ct < CT; ct++) {
            // m = -inf only in a column without a score yet
            const float refc = fmaxf(m[ct], -3.0e38f);
            float arg[4], vf[4], scaled[4];   // vf: the operands' V factors
            exp_args(dot_prev[ct], qsc[ct], ksr, refc, large, arg);
#pragma unroll
            for (int r = 0; r < 4; r++) vf[r] = vsr[r] * vinv[ct];
            if (edge)   // uniform. A token the row does not see may exceed vref by any factor: its vf too is 0
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const bool seen = t0 + r < row_end[ct];
                    arg[r] = seen ? arg[r] : -INFINITY;
                    vf[r] = seen ? vf[r] : 0.0f;
                }
            float total = 0.0f;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float prob = __builtin_amdgcn_exp2f(arg[r]);   // 0 for masked tokens
                total += prob;
                scaled[r] = prob * vf[r];
                // one rounded FP32 value: else the operand's hi is the exact product rounded once
                // (v_fma_mixlo_f16) and the hi that lo completes the rounded product rounded again,
                // which differ by 2^-10 in rare near-ties
                asm("" : "+v"(scaled[r]));
            }
            total_prev[ct] = total;
            half4 hi, lo;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                hi[r] = (_Float16)scaled[r];
                lo[r] = (_Float16)(scaled[r] - (float)hi[r]);
            }
            pshare[slot][ct][0][wave][n][qq] = __builtin_bit_cast(uint2, hi);
            pshare[slot][ct][1][wave][n][qq] = __builtin_bit_cast(uint2, lo);
        }
    };
#pragma unroll
    for (int e = 0; e < 16; e++) ow[e] = 0.0f;
    // the phases of decode_int8_kernel: finish chunk j - 1, score chunk j, stage V of chunk j and K of
    // chunk j + 1, load V of chunk j + 1 and K of chunk j + 2; one barrier each
    auto finish = [&](uint32_t j) __attribute__((always_inline)) {
        const int slot = (j - 1) & 1;
        float ctop[CT];
        bool raise = false;
#pragma unroll
        for (int ct = 0; ct < CT; ct++) {
            const float4 a = *reinterpret_cast<const float4 *>(&chunk_top[slot][ct][n][0]);
            const float4 b = *reinterpret_cast<const float4 *>(&chunk_top[slot][ct][n][4]);
            ctop[ct] = fmaxf(fmaxf(fmaxf(a.x, a.y), fmaxf(a.z, a.w)), fmaxf(fmaxf(b.x, b.y), fmaxf(b.z, b.w)));
            raise |= ctop[ct] > m[ct] + 8.0f;
        }
        // every wave reads the same maxima: the branch is uniform over the work-group. Only the
        // columns that passed the bound change (the others' factor is 1 and their operands the same).
        // Chunk 0 has no reference before its maxima: its operands are made here
        if (j == 1 || __builtin_amdgcn_ballot_w64(raise) != 0) {
            float decay[CT];
            bool any_large = false;
#pragma unroll
            for (int ct = 0; ct < CT; ct++) {
                const float next = ctop[ct] > m[ct] + 8.0f ? ctop[ct] : m[ct];
                decay[ct] = next == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m[ct] - next);
                l[ct] *= decay[ct];
                m[ct] = next;
                any_large |= large_ref(next);
            }
            large = __builtin_amdgcn_ballot_w64(any_large) != 0;
            if constexpr (kWide) {
                const float first = decay[0], second = decay[CT - 1];
                ow *= oct ? second : first;
            } else {
#pragma unroll
                for (int ct = 0; ct < CT; ct++) {
                    o[0][ct] *= decay[ct];
                    o[1][ct] *= decay[ct];
                }
            }
            probs(j - 1);
            __syncthreads();
        }
#pragma unroll
        for (int ct = 0; ct < CT; ct++) l[ct] += total_prev[ct];
        if constexpr (kWide) {
            // step s takes the 16 tokens of wave s: lane (column lane % 32, half lane / 32) 8 of them, P as
            // published, V in one 8-byte read of dimension 32 wave + lane % 32. Two MFMAs of 32 cycles a
            // step leave issue slots for its eight conversions (1000 + 476 keys and rows 40.3 -> 38.3
            // us against 16x16 tiles)
            const int half = lane >> 5, d = 32 * wave + (lane & 31);
            half8 ps[2][2];
            uint2 w8[2];
            auto read = [&](int s) __attribute__((always_inline)) {
#pragma unroll
                for (int hl = 0; hl < 2; hl++) ps[s & 1][hl] = *reinterpret_cast<const half8 *>(&pshare[slot][oct][hl][s][n][2 * half]);
                w8[s & 1] = reinterpret_cast<const uint2 *>(&vbuf[slot][d][s ^ ((d >> 1) & 7)])[half];
            };
            read(0);
#pragma unroll
            for (int s = 0; s < kDecodeWaves; s++) {
                if (s + 1 < kDecodeWaves) read(s + 1);
                uint32_t h0, h1, h2, h3;
                i8x8_to_f16_sdwa(w8[s & 1].x, w8[s & 1].y, h0, h1, h2, h3);
                const half8 va8 = __builtin_bit_cast(half8, make_uint4(h0, h1, h2, h3));
#pragma unroll
                for (int hl = 0; hl < 2; hl++) ow = __builtin_amdgcn_mfma_f32_32x32x16_f16(va8, ps[s & 1][hl], ow, 0, 0, 0);
            }
        } else {
            // step s takes the 32 tokens of waves 2s and 2s + 1, its operands read a step ahead
            half8 ps[2][CT][2];
            uint2 w8[2][2];
            auto read = [&](int s) __attribute__((always_inline)) {
                const int src = 2 * s + (qq >> 1);
#pragma unroll
                for (int ct = 0; ct < CT; ct++)
#pragma unroll
                    for (int hl = 0; hl < 2; hl++)
                        ps[s & 1][ct][hl] = *reinterpret_cast<const half8 *>(&pshare[slot][ct][hl][src][n][2 * (qq & 1)]);
#pragma unroll
                for (int dt = 0; dt < 2; dt++) {
                    const int d = 16 * (2 * wave + dt) + n;
                    w8[s & 1][dt] = reinterpret_cast<const uint2 *>(&vbuf[slot][d][src ^ ((d >> 1) & 7)])[qq & 1];
                }
            };
            read(0);
#pragma unroll
            for (int s = 0; s < kDecodeWaves / 2; s++) {
                if (s + 1 < kDecodeWaves / 2) read(s + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int dt = 0; dt < 2; dt++) {
                    uint32_t h0, h1, h2, h3;
                    i8x8_to_f16_sdwa(w8[s & 1][dt].x, w8[s & 1][dt].y, h0, h1, h2, h3);
                    const half8 va8 = __builtin_bit_cast(half8, make_uint4(h0, h1, h2, h3));
#pragma unroll
                    for (int hl = 0; hl < 2; hl++)
#pragma unroll
                        for (int ct = 0; ct < CT; ct++)
                            o[dt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va8, ps[s & 1][ct][hl], o[dt][ct], 0, 0, 0);
                }
            }
        }
    };
    for (uint32_t j = 0; j < nchunks; j++) {
        v4i kop[4];   // chunk j's K operands, this wave's own rows: read ahead of chunk j - 1's end
#pragma unroll
        for (int jj = 0; jj < 4; jj++) kop[jj] = __builtin_bit_cast(v4i, kbuf[wave][n][(4 * jj + qq) ^ n]);
        if (j > 0) finish(j);
        {
            v4i acc[CT][3], q3[2][CT];
#pragma unroll
            for (int ct = 0; ct < CT; ct++) {
#pragma unroll
                for (int part = 0; part < 3; part++) acc[ct][part] = v4i{0, 0, 0, 0};
                q3[0][ct] = q3lds[ct][0][16 * qq + (n ^ qq)];
            }
#pragma unroll
            for (int jj = 0; jj < 4; jj++) {
                if (jj < 3) {
#pragma unroll
                    for (int ct = 0; ct < CT; ct++) q3[(jj + 1) & 1][ct] = q3lds[ct][jj + 1][16 * qq + (n ^ (4 * jj + 4 + qq))];
                }
#pragma unroll
                for (int ct = 0; ct < CT; ct++) {
                    acc[ct][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(kop[jj], qi[ct][0][jj], acc[ct][0], 0, 0, 0);
                    acc[ct][1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(kop[jj], qi[ct][1][jj], acc[ct][1], 0, 0, 0);
                }
#pragma unroll
                for (int ct = 0; ct < CT; ct++)
                    acc[ct][2] = __builtin_amdgcn_mfma_i32_16x16x64_i8(kop[jj], q3[jj & 1][ct], acc[ct][2], 0, 0, 0);
            }
            const int local0 = (int)(j * kChunk) + 16 * wave + 4 * qq;   // token offset inside the split
            const uint32_t t0 = begin + (uint32_t)local0;
            const bool edge = begin + (j + 1) * kChunk > first_end;
            const float4 ks4 = *reinterpret_cast<const float4 *>(&kscale[local0]);
            const float ksr[4] = {ks4.x, ks4.y, ks4.z, ks4.w};
            float top[CT];
#pragma unroll
            for (int ct = 0; ct < CT; ct++) {
                float score[4];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    // 254 dot1 + dot2 is an exact integer (|dots| < 2^22) and the dot's unit 1 / 254. The
                    // exponent's argument is one fma of the dot (probs), so the score itself, rounded,
                    // is only compared
                    const float d12 = (float)(__mul24(acc[ct][0][r], 254) + acc[ct][1][r]);
                    dot_prev[ct][r] = fmaf((float)acc[ct][2][r], 1.0f / 254.0f, d12);
                    score[r] = dot_prev[ct][r] * (qsc[ct] * ksr[r]);
                }
                if (edge)
#pragma unroll
                    for (int r = 0; r < 4; r++) score[r] = t0 + r < row_end[ct] ? score[r] : -INFINITY;
                top[ct] = fmaxf(fmaxf(score[0], score[1]), fmaxf(score[2], score[3]));
            }
            // over the lanes of a column: with two tiles one swap of halves serves both, lanes below 32
            // ending with tile 0's maximum and the others with tile 1's
            float t = top[0];
            if constexpr (CT == 2) {
                float u = top[1];
                asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(t), "+v"(u));
                t = fmaxf(t, u);
            } else {
                t = xl_max32(t);
            }
            t = xl_max16(t);
            if ((qq & 1) == 0 && (CT == 2 || qq == 0)) chunk_top[j & 1][CT == 2 ? qq >> 1 : 0][n][wave] = t;
            if (j > 0) probs(j);
        }
        store_v(j & 1, rv);
        if (j + 1 < nchunks) {
            load_v(rv, j + 1);
            store_k(rk);
        }
        if (j + 2 < nchunks) load_k(rk, j + 2);
        __syncthreads();
    }
    finish(nchunks);

    // ---- O^T[d][n] times the column's V scale reference, l over the lanes and waves
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
        float lt = xl_sum32(xl_sum16(l[ct]));
        shift_large_values(vref[ct], lt, m[ct]);
        if (qq == 0) wave_l[ct][wave][n] = lt;
    }
    // the lane's quads of O, four dimensions of one column each: tile, first dimension, values
    constexpr int kQuads = kWide ? 4 : 2 * CT;
    auto quad_tile = [&](int u) __attribute__((always_inline)) { return kWide ? oct : u / 2; };
    auto quad_dim = [&](int u) __attribute__((always_inline)) {
        return 32 * wave + (kWide ? 8 * u + 4 * (lane >> 5) : 16 * (u % 2) + 4 * qq);
    };
    auto quad = [&](int u) __attribute__((always_inline)) {
        float v;
        floatx4 x;
        if constexpr (kWide) {
            const float first = vref[0], second = vref[CT - 1];
            v = oct ? second : first;
            x = floatx4{ow[4 * u], ow[4 * u + 1], ow[4 * u + 2], ow[4 * u + 3]};
        } else {
            v = vref[u / 2];
            x = o[u % 2][u / 2];
        }
        return make_float4(x[0] * v, x[1] * v, x[2] * v, x[3] * v);
    };
    if (p.splits > 1) {   // the partials' O needs no other wave's l
#pragma unroll
        for (int u = 0; u < kQuads; u++) {
            const uint32_t ri = 2 * quad_tile(u) + (n >> 3);
            if (ri < nr) *reinterpret_cast<float4 *>(part_of(ri) + head * 256 + quad_dim(u)) = quad(u);
        }
        __syncthreads();
        if (wave == 0 && qq == 0) {
#pragma unroll
            for (int ct = 0; ct < CT; ct++) {
                const uint32_t ri = 2 * ct + (n >> 3);
                if (ri >= nr) continue;
                float lw = 0.0f;
#pragma unroll
                for (int w = 0; w < kDecodeWaves; w++) lw += wave_l[ct][w][n];
                float *part = part_of(ri);
                part[2048 + head] = m[ct];
                part[2056 + head] = lw;
            }
        }
        return;
    }
    // gate and y need only 4-byte alignment; all gate loads go out before the first store (the
    // compiler cannot tell y from gate)
    float gate[kQuads][4];
    auto out_at = [&](int u) __attribute__((always_inline)) {
        const uint32_t row = r0 + min((uint32_t)(2 * quad_tile(u) + (n >> 3)), nr - 1);
        return ((size_t)row * 16 + g * 8 + head) * 256 + quad_dim(u);
    };
#pragma unroll
    for (int u = 0; u < kQuads; u++)
#pragma unroll
        for (int e = 0; e < 4; e++) gate[u][e] = p.gate[out_at(u) + e];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kQuads; u++) {
        float lw = 0.0f;
#pragma unroll
        for (int w = 0; w < kDecodeWaves; w++) lw += wave_l[quad_tile(u)][w][n];
        if ((uint32_t)(2 * quad_tile(u) + (n >> 3)) >= nr) continue;
        const float inv = 1.0f / lw;
        const float4 x = quad(u);
        float *at = p.y + out_at(u);
        at[0] = x.x * inv * sigmoidf(gate[u][0]);
        at[1] = x.y * inv * sigmoidf(gate[u][1]);
        at[2] = x.z * inv * sigmoidf(gate[u][2]);
        at[3] = x.w * inv * sigmoidf(gate[u][3]);
    }
}

inline bool aligned(const void *p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

}  // namespace

const char *launch_scores_int8(Context &c, const View *b, int count, const boot_kernel_args &p, const uint32_t *) {
    // bindings: q FP32 [rows][16][256], k INT8 cache, scores [rows][16][K], ks (QwenEngine.cs:163, Prefill.cs:280)
    BOOT_REQUIRE(count >= 4, "batch_attention_scores_int8 needs 4 bindings: q, k, scores, ks");
    const uint64_t rows = p.m, K = p.k;
    if (rows == 0 || K == 0) return nullptr;
    const uint64_t length = std::min<uint64_t>(K, (uint64_t)p.pos + rows);  // keys actually read
    BOOT_REQUIRE(b[0].bytes >= rows * 16384, "query buffer smaller than rows*4096 floats");
    BOOT_REQUIRE(b[1].bytes >= length * 512, "K cache smaller than the attended length");
    BOOT_REQUIRE(b[2].bytes >= rows * 16 * K * 4, "scores buffer smaller than rows*16*K floats");
    BOOT_REQUIRE(b[3].bytes >= length * 8, "K scale buffer smaller than the attended length");
    BOOT_REQUIRE(aligned(b[0].ptr, 4) && aligned(b[1].ptr, 16) && aligned(b[2].ptr, 4) && aligned(b[3].ptr, 4),
                 "bindings misaligned");
    // rows per work-group: the fewest of 1, 2, 4 that hold the dispatch's rows, at most 4 (an
    // 8-row work-group reads K once for all rows but holds one work-group per CU and streams
    // slower: 63.6 against 54.0 us at 8 rows over 131072 keys); a row's scores are the same in each
    const int per = rows >= 3 ? 4 : rows == 2 ? 2 : 1;
    const uint64_t zs = (rows + per - 1) / per;
    BOOT_REQUIRE(zs <= 65535, "batch_attention_scores_int8 serves at most 262140 rows");
    // tokens per work-group: 512 where the grid still holds four work-groups per CU (each one then
    // builds its rows' query operands for twice the tokens: 8 rows over 131072 keys 38.3 -> 32.7
    // us), else 256 (4 rows over 30000 keys: 12.5 us, against 18.1 with 512); a score does not
    // depend on the span
    const uint64_t wide = (K + 511) / 512;
    const uint32_t span = 2 * wide * zs >= 4 * (uint64_t)std::max(1, context_cus(c)) ? 512u : 256u;
    const uint64_t ktiles = (K + span - 1) / span;
    const dim3 sgrid((uint32_t)((2 * ktiles + 7) / 8 * 8 * zs));
    const float *qp = (const float *)b[0].ptr, *ksp = (const float *)b[3].ptr;
    const int8_t *kp = (const int8_t *)b[1].ptr;
    float *sp = (float *)b[2].ptr;
    if (per == 4)
        launch_timed(c, "scores_int8_kernel", scores_int8_kernel<4>, sgrid, dim3(256), qp, kp, sp, ksp, (uint32_t)rows,
                     (uint32_t)K, p.pos, (uint32_t)ktiles, (uint32_t)zs, span);
    else if (per == 2)
        launch_timed(c, "scores_int8_kernel", scores_int8_kernel<2>, sgrid, dim3(256), qp, kp, sp, ksp, (uint32_t)rows,
                     (uint32_t)K, p.pos, (uint32_t)ktiles, (uint32_t)zs, span);
    else
        launch_timed(c, "scores_int8_kernel", scores_int8_kernel<1>, sgrid, dim3(256), qp, kp, sp, ksp, (uint32_t)rows,
                     (uint32_t)K, p.pos, (uint32_t)ktiles, (uint32_t)zs, span);
    return nullptr;
}

const char *launch_softmax(Context &c, const View *b, int count, const boot_kernel_args &p, const uint32_t *grid) {
    // bindings: x scores [groups][K]; groups = dispatched threads / 256 (QwenEngine.cs:164, Prefill.cs:282)
    BOOT_REQUIRE(count >= 1, "attention_softmax needs 1 binding: scores");
    BOOT_REQUIRE(grid[3] == 256 && grid[1] <= 1 && grid[2] <= 1, "attention_softmax is dispatched as groups of 256 threads");
    const uint64_t groups = grid[0] / 256, K = p.k;
    if (groups == 0) return nullptr;
    BOOT_REQUIRE(p.pos < K, "softmax position must be below the row stride K");
    BOOT_REQUIRE(b[0].bytes >= groups * K * 4, "scores buffer smaller than groups*K floats");
    BOOT_REQUIRE(aligned(b[0].ptr, 4), "scores binding misaligned");
    // chunk statistics of every row, then each chunk normalized with its row's merged statistics
    const uint64_t chunks = ((uint64_t)p.pos + 1 + kSoftmaxChunk - 1) / kSoftmaxChunk;
    BOOT_REQUIRE(groups <= 65535, "attention_softmax serves at most 65535 rows");
    float2 *stats = (float2 *)context_workspace(c, groups * chunks * sizeof(float2));
    BOOT_REQUIRE(stats, "cannot allocate softmax workspace");
    const dim3 sgrid((uint32_t)chunks, (uint32_t)groups);
    launch_timed(c, "softmax_stats_kernel", softmax_stats_kernel, sgrid, dim3(256), (const float *)b[0].ptr, stats,
                 (uint32_t)K, p.pos, (uint32_t)chunks);
    launch_timed(c, "softmax_apply_kernel", softmax_apply_kernel, sgrid, dim3(256), (float *)b[0].ptr,
                 (const float2 *)stats, (uint32_t)K, p.pos, (uint32_t)chunks);
    return nullptr;
}

const char *launch_values_int8(Context &c, const View *b, int count, const boot_kernel_args &p, const uint32_t *) {
    // bindings: scores, v INT8 pages, gate, y, vs (QwenEngine.cs:165, Prefill.cs:283)
    BOOT_REQUIRE(count >= 5, "batch_attention_values_int8 needs 5 bindings: scores, v, gate, y, vs");
    const uint64_t rows = p.m, K = p.k;
    if (rows == 0) return nullptr;
    BOOT_REQUIRE(rows <= 65535, "batch_attention_values_int8 serves at most 65535 rows");   // the combine's grid
    const uint64_t length = (uint64_t)p.pos + rows;
    BOOT_REQUIRE(length <= K, "causal end pos+rows exceeds the score row stride K");
    BOOT_REQUIRE(b[0].bytes >= rows * 16 * K * 4, "scores buffer smaller than rows*16*K floats");
    BOOT_REQUIRE(b[1].bytes >= value_bytes(length), "V cache smaller than whole pages of the attended length");
    BOOT_REQUIRE(b[2].bytes >= rows * 16384 && b[3].bytes >= rows * 16384, "gate/output smaller than rows*4096 floats");
    BOOT_REQUIRE(b[4].bytes >= length * 8, "V scale buffer smaller than the attended length");
    BOOT_REQUIRE(aligned(b[1].ptr, 16), "V cache binding must be 16-byte aligned");
    // split partials over absolute kValuesSplit-token ranges, then their sum in order with the gate
    const uint64_t splits = (K + kValuesSplit - 1) / kValuesSplit;
    float *part = (float *)context_workspace(c, rows * 2 * splits * 2048 * sizeof(float));
    BOOT_REQUIRE(part, "cannot allocate values workspace");
    // rows per work-group: the fewest of 1, 2, 4 that hold the dispatch's rows, at most 4 (8 rows
    // take 276 registers, one work-group per CU: 74.0 against 52.2 us at 8 rows over 131072 keys;
    // 2 rows read V four times: 63.6 us); a row's result is the same in each
    const int per = rows >= 3 ? 4 : rows == 2 ? 2 : 1;
    const uint64_t zs = (rows + per - 1) / per;
    const dim3 vgrid((uint32_t)((2 * splits + 7) / 8 * 8 * zs));
    const float *sc = (const float *)b[0].ptr, *vsc = (const float *)b[4].ptr;
    const int8_t *vc = (const int8_t *)b[1].ptr;
    if (per == 4)
        launch_timed(c, "values_partial_kernel", values_partial_kernel<4>, vgrid, dim3(512), sc, vc, vsc, part,
                     (uint32_t)rows, (uint32_t)K, p.pos, (uint32_t)splits, (uint32_t)zs);
    else if (per == 2)
        launch_timed(c, "values_partial_kernel", values_partial_kernel<2>, vgrid, dim3(512), sc, vc, vsc, part,
                     (uint32_t)rows, (uint32_t)K, p.pos, (uint32_t)splits, (uint32_t)zs);
    else
        launch_timed(c, "values_partial_kernel", values_partial_kernel<1>, vgrid, dim3(512), sc, vc, vsc, part,
                     (uint32_t)rows, (uint32_t)K, p.pos, (uint32_t)splits, (uint32_t)zs);
    launch_timed(c, "values_combine_kernel", values_combine_kernel, dim3(64, (uint32_t)rows), dim3(64),
                 (const float *)part, (const float *)b[2].ptr, (float *)b[3].ptr, (uint32_t)splits);
    return nullptr;
}

namespace {

// Split geometry shared by both decode entry points: whole 128-token chunks per split, chosen so
// that the grid (splits x 2 groups x rows, one work-group per CU) fits the CUs in one round (a
// second, nearly empty round would double the time), at most kMaxSplitTokens per split. Two chunks
// stay in one split: the second chunk takes less than the combine's launch, which falls away (ten
// layers' token after 128 to 255 tokens 115-121 us in two splits, 101-106 in one); three chunks
// measure the same either way (119-121 us after 256 to 383 tokens).
template <bool kHalfQ = false>
const char *decode_launch(Context &c, DecodeParams &d, uint64_t rows, uint64_t length) {
    const uint64_t total_chunks = (length + kChunk - 1) / kChunk;
    const uint64_t slots = std::max<uint64_t>(1, (uint64_t)std::max(1, context_cus(c)) / (2 * rows));
    uint64_t split_chunks = (total_chunks + slots - 1) / slots;
    split_chunks = std::min<uint64_t>(split_chunks, (uint64_t)(kMaxSplitTokens / kChunk));
    if (total_chunks == 2) split_chunks = 2;
    const uint64_t splits = (total_chunks + split_chunks - 1) / split_chunks;
    BOOT_REQUIRE(splits <= kMaxDecodeSplits, "too many decode splits");
    d.rows = (uint32_t)rows;
    d.splits = (uint32_t)splits;
    d.split_chunks = (uint32_t)split_chunks;
    d.partial = nullptr;
    if (splits > 1) {
        d.partial = (float *)context_workspace(c, rows * 2 * splits * kPartialFloats * sizeof(float));
        BOOT_REQUIRE(d.partial, "cannot allocate decode split workspace");
    }
    launch_timed(c, kHalfQ ? "decode_int8_half_query_kernel" : "decode_int8_kernel", decode_int8_kernel<kHalfQ>,
                 dim3((uint32_t)splits, 2, (uint32_t)rows), dim3(512), d);
    if (splits > 1) {
        context_split(c, "attention_decode_int8.combine");
        launch_timed(c, "decode_combine_kernel", decode_combine_kernel, dim3(4, 16, (uint32_t)rows), dim3(256), d.partial,
                     d.gate, d.y, (uint32_t)splits);
    }
    return nullptr;
}

}  // namespace

const char *launch_decode_append_int8(Context &c, const View *b, int count, const boot_kernel_args &p,
                                      const uint32_t *) {
    // bindings: q FP32 [1][16][256] (unrotated), k, v FP32 [1][2][256] (the new token, K
    // unrotated), rotated FP32 [1][16][256] (out), kc, vc, ks, vs (the cache, appended at
    // Position), gate, y. One decode step of QwenEngine.cs:161-165: batch_rope_int8 with M = 1
    // followed by attention over keys 0..Position, in one dispatch.
    BOOT_REQUIRE(count >= 10, "attention_decode_append_int8 needs 10 bindings: q, k, v, rotated, kc, vc, ks, vs, gate, y");
    BOOT_REQUIRE(p.m == 1, "attention_decode_append_int8 serves one row (M = 1)");
    const uint64_t length = (uint64_t)p.pos + 1;
    BOOT_REQUIRE(length <= 262144, "attended length exceeds the 262144-token window");
    BOOT_REQUIRE(b[0].bytes >= 16384 && b[3].bytes >= 16384, "query/rotated buffers smaller than 4096 floats");
    BOOT_REQUIRE(b[1].bytes >= 2048 && b[2].bytes >= 2048, "K/V input smaller than 512 floats");
    BOOT_REQUIRE(b[4].bytes >= length * 512, "K cache smaller than Position + 1 tokens");
    BOOT_REQUIRE(b[5].bytes >= value_bytes(length), "V cache smaller than whole pages of Position + 1 tokens");
    BOOT_REQUIRE(b[6].bytes >= length * 8 && b[7].bytes >= length * 8, "KV scale buffers smaller than Position + 1 tokens");
    BOOT_REQUIRE(b[8].bytes >= 16384 && b[9].bytes >= 16384, "gate/output smaller than 4096 floats");
    BOOT_REQUIRE(aligned(b[0].ptr, 16) && aligned(b[1].ptr, 16) && aligned(b[2].ptr, 16) && aligned(b[3].ptr, 16) &&
                     aligned(b[4].ptr, 16) && aligned(b[5].ptr, 16) && aligned(b[6].ptr, 4) && aligned(b[7].ptr, 4) &&
                     aligned(b[8].ptr, 4) && aligned(b[9].ptr, 4),
                 "bindings misaligned (q, k, v, rotated, kc, vc need 16 bytes)");
    DecodeParams d;
    d.q = (const float *)b[0].ptr;
    d.qh = nullptr;
    d.knew = (const float *)b[1].ptr;
    d.vnew = (const float *)b[2].ptr;
    d.rotated = (float *)b[3].ptr;
    d.k = (const int8_t *)b[4].ptr;
    d.v = (const int8_t *)b[5].ptr;
    d.ks = (const float *)b[6].ptr;
    d.vs = (const float *)b[7].ptr;
    d.k_out = (int8_t *)b[4].ptr;
    d.v_out = (int8_t *)b[5].ptr;
    d.ks_out = (float *)b[6].ptr;
    d.vs_out = (float *)b[7].ptr;
    d.gate = (const float *)b[8].ptr;
    d.y = (float *)b[9].ptr;
    d.pos = p.pos;
    d.append = 1;
    d.freq = context_rope(c, p.theta);
    return decode_launch(c, d, 1, length);
}

const char *launch_decode_int8(Context &c, const View *b, int count, const boot_kernel_args &p, const uint32_t *) {
    // bindings (EncodeInt8 order, DeviceAttention.cs:69): q FP32 [rows][16][256] (rotated),
    // k, v, gate, y, ks, vs. Row r attends t <= pos + r.
    BOOT_REQUIRE(count >= 7, "attention_decode_int8 needs 7 bindings: q, k, v, gate, y, ks, vs");
    const uint64_t rows = p.m;
    if (rows == 0) return nullptr;
    BOOT_REQUIRE(rows <= 64, "attention_decode_int8 serves at most 64 rows");
    const uint64_t length = (uint64_t)p.pos + rows;
    BOOT_REQUIRE(length <= 262144, "attended length exceeds the 262144-token window");
    BOOT_REQUIRE(b[0].bytes >= rows * 16384, "query buffer smaller than rows*4096 floats");
    BOOT_REQUIRE(b[1].bytes >= length * 512, "K cache smaller than the attended length");
    BOOT_REQUIRE(b[2].bytes >= value_bytes(length), "V cache smaller than whole pages of the attended length");
    BOOT_REQUIRE(b[3].bytes >= rows * 16384 && b[4].bytes >= rows * 16384, "gate/output smaller than rows*4096 floats");
    BOOT_REQUIRE(b[5].bytes >= length * 8 && b[6].bytes >= length * 8, "KV scale buffers smaller than the attended length");
    BOOT_REQUIRE(aligned(b[0].ptr, 16) && aligned(b[1].ptr, 16) && aligned(b[2].ptr, 16) && aligned(b[3].ptr, 4) &&
                     aligned(b[4].ptr, 4) && aligned(b[5].ptr, 4) && aligned(b[6].ptr, 4),
                 "bindings misaligned (q, k, v need 16 bytes)");
    DecodeParams d;
    d.q = (const float *)b[0].ptr;
    d.qh = nullptr;
    d.k = (const int8_t *)b[1].ptr;
    d.v = (const int8_t *)b[2].ptr;
    d.gate = (const float *)b[3].ptr;
    d.y = (float *)b[4].ptr;
    d.ks = (const float *)b[5].ptr;
    d.vs = (const float *)b[6].ptr;
    d.pos = p.pos;
    d.append = 0;
    d.freq = RopeFreq{};
    d.knew = d.vnew = nullptr;
    d.rotated = nullptr;
    d.k_out = d.v_out = nullptr;
    d.ks_out = d.vs_out = nullptr;
    return decode_launch(c, d, rows, length);
}

const char *launch_verify_int8(Context &c, const View *b, int count, const boot_kernel_args &p, const uint32_t *) {
    // bindings (attention_decode_int8's order): q FP32 [rows][16][256] (rotated), k, v, gate, y, ks, vs.
    // Row r attends t <= pos + r; its result depends on that row alone, and y may be q.
    BOOT_REQUIRE(count >= 7, "attention_verify_int8 needs 7 bindings: q, k, v, gate, y, ks, vs");
    const uint64_t rows = p.m;
    if (rows == 0) return nullptr;
    BOOT_REQUIRE(rows <= 64, "attention_verify_int8 serves at most 64 rows");
    const uint64_t length = (uint64_t)p.pos + rows;
    BOOT_REQUIRE(length <= 262144, "attended length exceeds the 262144-token window");
    BOOT_REQUIRE(b[0].bytes >= rows * 16384, "query buffer smaller than rows*4096 floats");
    BOOT_REQUIRE(b[1].bytes >= length * 512, "K cache smaller than the attended length");
    BOOT_REQUIRE(b[2].bytes >= value_bytes(length), "V cache smaller than whole pages of the attended length");
    BOOT_REQUIRE(b[3].bytes >= rows * 16384 && b[4].bytes >= rows * 16384, "gate/output smaller than rows*4096 floats");
    BOOT_REQUIRE(b[5].bytes >= length * 8 && b[6].bytes >= length * 8, "KV scale buffers smaller than the attended length");
    BOOT_REQUIRE(aligned(b[0].ptr, 16) && aligned(b[1].ptr, 16) && aligned(b[2].ptr, 16) && aligned(b[3].ptr, 4) &&
                     aligned(b[4].ptr, 4) && aligned(b[5].ptr, 4) && aligned(b[6].ptr, 4),
                 "bindings misaligned (q, k, v need 16 bytes)");
    // A row's split is as many chunks as spread its own keys over a number of work-groups per KV
    // group, whatever rows come with it, so that its result depends on its position alone; rows of
    // one launch have the same split (a block across a boundary takes two launches). 64 work-groups
    // up to 65536 keys: with two groups and two row blocks one round of 256 CUs, 8 rows after 9000
    // keys 19.4 (128 work-groups: 27.8) us, after 30000 24.7 (35.0), where 4 rows lose little, 18.6
    // (17.3) and 24.4 (24.1) us. 128 beyond, one round for up to 4 rows: 100000 keys 38.4 (64: 46.9)
    // us, against 63.4 (48.5) us for 8 rows.
    constexpr uint32_t kNearChunks = 65536 / kChunk, kNearSlots = 64, kFarSlots = 128;
    auto chunks_of = [&](uint64_t row) { return (uint32_t)(((uint64_t)p.pos + row) / kChunk + 1); };
    auto split_of = [&](uint64_t row) {
        const uint32_t chunks = chunks_of(row), slots = chunks <= kNearChunks ? kNearSlots : kFarSlots;
        return (chunks + slots - 1) / slots;
    };
    static_assert(kNearChunks <= kNearSlots * (kMaxSplitTokens / kChunk) &&
                      262144 / kChunk <= kFarSlots * (kMaxSplitTokens / kChunk), "a split's scales exceed the LDS");
    // one past the last row of the launch that starts with row `first`, and that launch's splits
    auto launch_end = [&](uint64_t first) {
        uint64_t next = first + 1;
        while (next < rows && split_of(next) == split_of(first)) next++;
        return next;
    };
    auto splits_of = [&](uint64_t first, uint64_t next) {
        const uint32_t per = split_of(first);
        return (chunks_of(next - 1) + per - 1) / per;
    };
    // The scratch of the largest launch, before the first one: y may be q, so a request refused after a
    // launch would leave some queries overwritten.
    uint64_t scratch = 0;
    for (uint64_t first = 0, next; first < rows; first = next) {
        next = launch_end(first);
        const uint64_t splits = splits_of(first, next);
        if (splits > 1) scratch = std::max<uint64_t>(scratch, (next - first) * 2 * splits * kPartialFloats * sizeof(float));
    }
    float *partial = nullptr;
    if (scratch) {
        partial = (float *)context_workspace(c, scratch);
        BOOT_REQUIRE(partial, "cannot allocate verify split workspace");
    }
    for (uint64_t first = 0, next; first < rows; first = next) {
        next = launch_end(first);
        RowsParams d;
        d.qh = nullptr;
        d.q = (const float *)b[0].ptr + first * 4096;
        d.k = (const int8_t *)b[1].ptr;
        d.v = (const int8_t *)b[2].ptr;
        d.gate = (const float *)b[3].ptr + first * 4096;
        d.y = (float *)b[4].ptr + first * 4096;
        d.ks = (const float *)b[5].ptr;
        d.vs = (const float *)b[6].ptr;
        d.rows = (uint32_t)(next - first);
        d.pos = (uint32_t)(p.pos + first);
        d.split_chunks = split_of(first);
        d.splits = splits_of(first, next);
        d.partial = d.splits > 1 ? partial : nullptr;
        // one or two rows: half the columns and registers (1 row after 1500 keys 7.8 against 9.7 us)
        const bool narrow = d.rows <= 2;
        d.zs = narrow ? 1 : (d.rows + 3) / 4;
        const dim3 grid((2 * d.splits + 7) / 8 * 8 * d.zs);
        launch_timed(c, "rows_int8_kernel",
                     narrow        ? rows_int8_kernel<1, true, false>
                     : d.zs == 1 ? rows_int8_kernel<2, true, false>
                                 : rows_int8_kernel<2, false, false>,
                     grid, dim3(512), d);
        if (d.splits > 1)
            launch_timed(c, "decode_combine_kernel", decode_combine_kernel, dim3(4, 16, d.rows), dim3(256),
                         (const float *)d.partial, d.gate, d.y, d.splits);
    }
    return nullptr;
}

const char *launch_online_int8_as_decode(Context &c, const View *b, const boot_kernel_args &p) {
    // A prefill chunk of at most 64 rows over a short history (launch_prefill's choice, which has
    // validated the bindings: grouped FP16 q, k, v, gate, y, ks, vs): one work-group per (row, KV
    // group, split) streams the keys up to its own row's position, as a decode of that many rows,
    // instead of 256-row tiles that are mostly empty.
    const uint64_t rows = p.m, length = (uint64_t)p.pos + rows;
    BOOT_REQUIRE(rows >= 1 && rows <= 64, "a prefill chunk served by the decode kernel has 1 to 64 rows");
    DecodeParams d;
    d.q = nullptr;
    d.qh = (const _Float16 *)b[0].ptr;
    d.k = (const int8_t *)b[1].ptr;
    d.v = (const int8_t *)b[2].ptr;
    d.gate = (const float *)b[3].ptr;
    d.y = (float *)b[4].ptr;
    d.ks = (const float *)b[5].ptr;
    d.vs = (const float *)b[6].ptr;
    d.pos = p.pos;
    d.append = 0;
    d.freq = RopeFreq{};
    d.knew = d.vnew = nullptr;
    d.rotated = nullptr;
    d.k_out = d.v_out = nullptr;
    d.ks_out = d.vs_out = nullptr;
    return decode_launch<true>(c, d, rows, length);
}

const char *launch_online_int8_rows(Context &c, const View *b, const boot_kernel_args &p) {
    // A prefill chunk on rows_int8_kernel (launch_prefill's choice, which has validated the bindings:
    // grouped FP16 q, k, v, gate, y, ks, vs).
    const uint64_t rows = p.m, length = (uint64_t)p.pos + rows;
    BOOT_REQUIRE(rows >= 1 && rows <= 512, "a prefill chunk served by the multi-row kernel has 1 to 512 rows");
    RowsParams d;
    d.q = nullptr;
    d.qh = (const _Float16 *)b[0].ptr;
    d.k = (const int8_t *)b[1].ptr;
    d.v = (const int8_t *)b[2].ptr;
    d.gate = (const float *)b[3].ptr;
    d.y = (float *)b[4].ptr;
    d.ks = (const float *)b[5].ptr;
    d.vs = (const float *)b[6].ptr;
    d.rows = (uint32_t)rows;
    d.pos = p.pos;
    d.zs = (uint32_t)((rows + 3) / 4);
    // One split, or one round of work-groups: a chunk of 128 keys takes about 2.5 us of a work-group,
    // the combine 4 us and 0.067 us per row (64 rows after 200 keys: 3 splits 18.0, one 15.2 us; 8
    // rows after 1000: 8 splits 14.0 us, one about 27). More than 64 rows are never split (the
    // combine of 200 rows takes 21 us).
    const uint64_t chunks = (length + kChunk - 1) / kChunk;
    const uint64_t slots = rows > 64 ? 1 : std::max<uint64_t>(1, (uint64_t)std::max(1, context_cus(c)) / (2 * d.zs));
    const uint64_t most = kMaxSplitTokens / kChunk, spread = std::min<uint64_t>((chunks + slots - 1) / slots, most);
    const uint64_t split_chunks = 24 * (chunks - spread) <= 40 + 2 * rows / 3 && chunks <= most ? chunks : spread;
    d.split_chunks = (uint32_t)split_chunks;
    d.splits = (uint32_t)((chunks + split_chunks - 1) / split_chunks);
    d.partial = nullptr;
    if (d.splits > 1) {
        d.partial = (float *)context_workspace(c, rows * 2 * d.splits * kPartialFloats * sizeof(float));
        BOOT_REQUIRE(d.partial, "cannot allocate prefill split workspace");
    }
    launch_timed(c, "rows_int8_half_query_kernel", rows_int8_kernel<2, false, true>, dim3(2 * d.splits * d.zs), dim3(512), d);
    if (d.splits > 1) {
        context_split(c, "attention_online_int8.combine");
        launch_timed(c, "decode_combine_kernel", decode_combine_kernel, dim3(4, 16, d.rows), dim3(256),
                     (const float *)d.partial, d.gate, d.y, d.splits);
    }
    return nullptr;
}

}  // namespace boot
