// The passes of the Hadamard MLP's Kronecker products on the f32 matrix cores
// (the layer kernel's, and nh_check.hip's over given operands).
#pragma once

#include "nh_device.h"
#include "nh_forward.h"

namespace nh {
namespace {

constexpr int MIX_T = 256;    // threads of one mix8: four wavefronts, a 16 x 16 tile of the output each
constexpr int BT_PITCH = 36;  // floats per row of a first mix8's output (16-byte reads; rows 4 banks apart)

// mix8 (infer.rs:2343-2380), portable branch: out[r][c] =
// sum_j ct[j][r] * rows[j][c] over 32 x 32, each output an fma chain from
// j = 0.  v_mfma_f32_16x16x4_f32 runs exactly that chain: its four products
// of an output are added one after the other in k order with one rounding
// each (bit-identical to the fmaf chain over random, wide-range, signed-zero,
// subnormal and non-finite operands: tests/test_gpu_mix8.py), so eight of
// them in j order are the reference's 32 steps.  Four wavefronts take a 16 x 16 tile of the output each.  A pass is
// one chain of eight dependent MFMAs (34 cycles each) between two LDS round
// trips, and a lane reads 8 + 8 operands for its 4 outputs; the same chains
// on the vector ALU (2 x 2 outputs a thread, 64 + 64 operands read for 4
// outputs) were bound by LDS bandwidth.  With cond_weights' conversions apart
// from its chain: 32 greedy tokens after a 118-token prompt 16.93 -> 16.58
// ms, a 512-token prefill 1.328 -> 1.313 ms.
//
// Lane (q, i) = (lane / 16, lane % 16) supplies factor element [4 s + q][16 tile + i]
// of step s, f16 in the staged fragment order: kf[tile * 64 + lane] holds
// s = 0..7 (the same element as operand A of the transposed pass, where
// the tile is the output's row block, and as operand B of the plain one,
// where it is its column block), and gets out[4 q + v][i] of its tile.
__device__ __forceinline__ f32x4 mix_chain(const uint4& f, const float (&x)[8], bool factor_rows) {
    const uint32_t fw[4] = {f.x, f.y, f.z, f.w};
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        const float k = f16_bits_to_f32((uint16_t)(fw[s >> 1] >> (16 * (s & 1))));
        acc = factor_rows ? __builtin_amdgcn_mfma_f32_16x16x4f32(k, x[s], acc, 0, 0, 0)
                          : __builtin_amdgcn_mfma_f32_16x16x4f32(x[s], k, acc, 0, 0, 0);
    }
    return acc;
}

// Element t (row j = t / 32, column c = t % 32) of the transposed pass's
// vector operand, column block major: a wavefront's reads of four rows x 16
// columns are 64 consecutive floats.
__device__ __forceinline__ int mix_in(int t) { return ((t >> 4) & 1) * (HADA_N / 2) + (t >> 5) * 16 + (t & 15); }

// Transposed (ct = a factor, rows = the vector operand in mix_in order):
// out[r][c] at out[r * BT_PITCH + 8 (c % 4) + c / 4], so that a lane of the
// plain pass reads its eight k elements as two 16-byte vectors.
__device__ __forceinline__ void mix8_t(int u, const uint4* kf, const float* rows, float* out) {
    const int lane = u & 63, q = lane >> 4, i = lane & 15, rt = (u >> 6) & 1, ct = u >> 7;
    const uint4 f = kf[rt * 64 + lane];
    float x[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) x[s] = rows[ct * (HADA_N / 2) + s * 64 + lane];
    const f32x4 o = mix_chain(f, x, true);
    const int c = ct * 16 + i;
#pragma unroll
    for (int v = 0; v < 4; ++v) out[(rt * 16 + 4 * q + v) * BT_PITCH + (c & 3) * 8 + (c >> 2)] = o[v];
}

// Plain (ct = the output of mix8_t, rows = a factor): out[r][c] row-major,
// rows r < rows_limit (a multiple of 8).
__device__ __forceinline__ void mix8_n(int u, const float* ct, const uint4* kf, float* out, int rows_limit) {
    const int lane = u & 63, q = lane >> 4, i = lane & 15, rt = (u >> 6) & 1, cb = u >> 7;
    const uint4 f = kf[cb * 64 + lane];
    const float4* xr = reinterpret_cast<const float4*>(ct + (rt * 16 + i) * BT_PITCH + q * 8);
    const float4 x0 = xr[0], x1 = xr[1];
    const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
    const f32x4 o = mix_chain(f, x, false);
    const int r = rt * 16 + 4 * q;
    if (r < rows_limit) {
#pragma unroll
        for (int v = 0; v < 4; ++v) out[(r + v) * HADA_NB + cb * 16 + i] = o[v];
    }
}

}  // namespace
}  // namespace nh
