// Fused RMSNorm -> 128-point FWHT -> int8 activation quantizer (A8).
//
// With a norm scale, a row's zero-centred RMSNorm comes first: ss =
// dot16(x, x) in the reference's accumulator order
// (crates/needle-engine/src/infer.rs:369-419, portable branch 401-418), r =
// 1 / sqrtf(ss / n + 1e-6) (infer.rs:422-424) and h = fma(x * r, s, x * r)
// (norm_apply16, infer.rs:614-635).  Then every 128-group is rotated
// (crates/needle-core/src/quant.rs:109-115) and quantized
// (crates/needle-engine/src/qlinear.rs:77-88, 152-164).  The int8 codes are
// written in the GEMV/GEMM activation order (act_offset), not the
// reference's act_pos order: the integer sums they feed are order-free, and
// nh_qact_download restores act_pos for checks.
//
// Many rows are bound by vector instructions, few by latency.  A lane holds
// 16 consecutive positions of a group, eight lanes a group, eight groups a
// wavefront: four of the FWHT's seven stages then stay inside a lane and the
// other three are DPP moves, a third of the instructions of two positions a
// lane (a8_group), and a lane's codes leave as two 8-byte stores (4-bit
// order) or one of 16 bytes (2-bit).  Graph replay, us, before (a workgroup
// a row, two positions a lane) and now: 4096 x 768 7.10 -> 4.16, with the
// norm 9.70 -> 6.25; 1024 x 3072 7.41 -> 4.03, 10.90 -> 8.99; 512 x 768
// 2.82 -> 2.50, 4.19 -> 4.14.
#include <algorithm>

#include "nh_device.h"
#include "nh_internal.h"

namespace nh {

constexpr int EL = 16;              // positions of a lane
constexpr int GL = GROUP / EL;      // lanes of a group
constexpr int ACT_WAVE = 64 / GL;   // groups of a wavefront

// The value of lane (lane ^ h), h = 1, 2 or 4, by DPP (4: the mirror within
// eight lanes, then the mirror within four).
template <int H>
__device__ __forceinline__ float oct_xor(float v) {
    const int b = __builtin_bit_cast(int, v);
    if constexpr (H == 1) return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, b, 0xB1, 0xF, 0xF, false));
    if constexpr (H == 2) return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, b, 0x4E, 0xF, 0xF, false));
    const int m = __builtin_amdgcn_update_dpp(0, b, 0x141, 0xF, 0xF, false);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, m, 0x1B, 0xF, 0xF, false));
}

// One cross-lane FWHT stage: a + b in the lower lane, a - b in the upper.
// fma(v, -1, p) is p - v rounded once.
template <int H>
__device__ __forceinline__ void oct_stage(float (&v)[EL], int l) {
    const float s = (l & H) ? -1.0f : 1.0f;
#pragma unroll
    for (int i = 0; i < EL; ++i) v[i] = __builtin_fmaf(v[i], s, oct_xor<H>(v[i]));
}

// prep_group of the group held by lanes 8 u + l, l < 8 (positions 16 l ..):
// codes to the group's 128-byte block `q`, the scale to `s_out`, stored by
// the lanes with `on`.
__device__ __forceinline__ void a8_oct(float (&v)[EL], int l, int bits, bool on, int8_t* q, float* s_out) {
#pragma unroll
    for (int h = 1; h < EL; h <<= 1)
#pragma unroll
        for (int i = 0; i < EL; ++i)
            if ((i & h) == 0) {
                const float a = v[i], b = v[i + h];
                v[i] = a + b;
                v[i + h] = a - b;
            }
    oct_stage<1>(v, l);
    oct_stage<2>(v, l);
    oct_stage<4>(v, l);
    const float hs = bits_f32(0x3db504f3u);
    // A maximum that keeps a NaN (v_maximum3_f32, at fmaxf's rate).
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < EL; ++i) {
        v[i] *= hs;
        m = __builtin_elementwise_maximum(m, fabsf(v[i]));
    }
    m = __builtin_elementwise_maximum(m, oct_xor<1>(m));
    m = __builtin_elementwise_maximum(m, oct_xor<2>(m));
    m = __builtin_elementwise_maximum(m, oct_xor<4>(m));
    // Non-finite inputs, and finite ones that overflow, leave NaNs in a group.
    // As in a8_group, one at both positions p and p + 64 makes the scale 1
    // (also where the other positions are finite); one whose partner is not
    // NaN is passed over by the maximum.
    if (__any(m != m)) {
        int both = 0;
        float mx = 0.0f;
#pragma unroll
        for (int i = 0; i < EL; ++i) {
            const float o = oct_xor<4>(v[i]);
            both |= (v[i] != v[i]) & (o != o);
            mx = fmaxf(mx, fabsf(v[i]));
        }
        float f = both ? 1.0f : 0.0f;
        f = fmaxf(f, oct_xor<1>(f));
        f = fmaxf(f, oct_xor<2>(f));
        f = fmaxf(f, oct_xor<4>(f));
        mx = fmaxf(mx, oct_xor<1>(mx));
        mx = fmaxf(mx, oct_xor<2>(mx));
        mx = fmaxf(mx, oct_xor<4>(mx));
        if (m != m) m = f != 0.0f ? 0.0f : mx;
    }
    const float s = m > 0.0f ? m * bits_f32(0x3c010204u) : 1.0f;
    const float inv = 1.0f / s;
    uint32_t w[EL / 4];
    // the positions of byte b of dword k: 4-bit, 8-position block k / 2, its
    // even positions then its odd ones; 2-bit, field k of byte b
#pragma unroll
    for (int k = 0; k < EL / 4; ++k) {
        uint32_t x = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const float e = bits == 2 ? v[4 * b + k] : v[(k >> 1) * 8 + 2 * b + (k & 1)];
            x |= (uint32_t)(uint8_t)quant_one(e, inv) << (8 * b);
        }
        w[k] = x;
    }
    if (on) {
        if (bits == 2) {
            *reinterpret_cast<uint4*>(q + act_offset(l * EL, 2)) = make_uint4(w[0], w[1], w[2], w[3]);
        } else {
            *reinterpret_cast<uint2*>(q + act_offset(l * EL, 4)) = make_uint2(w[0], w[1]);
            *reinterpret_cast<uint2*>(q + act_offset(l * EL + 8, 4)) = make_uint2(w[2], w[3]);
        }
        if (l == 0) *s_out = s;
    }
}

// A lane's 16 positions of a row from p0 on, zero from in_dim on.  vec: the
// rows are 16-byte aligned (the pointer, and in_dim a multiple of 4).
__device__ __forceinline__ void load_el(float (&v)[EL], const float* row, int p0, int in_dim, bool vec) {
    if (vec) {
#pragma unroll
        for (int i = 0; i < EL / 4; ++i) {
            const int p = p0 + 4 * i;
            const float4 f = p < in_dim ? *reinterpret_cast<const float4*>(row + p) : make_float4(0, 0, 0, 0);
            v[4 * i] = f.x, v[4 * i + 1] = f.y, v[4 * i + 2] = f.z, v[4 * i + 3] = f.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < EL; ++i) v[i] = p0 + i < in_dim ? row[p0 + i] : 0.0f;
    }
}

template <int BITS>
__global__ __launch_bounds__(64) void k_act_a8(const float* __restrict__ x, unsigned units, int in_dim, unsigned groups,
                                               int vec, int8_t* __restrict__ xq, float* __restrict__ sx) {
    const int lane = threadIdx.x, l = lane & (GL - 1);
    const unsigned unit = blockIdx.x * ACT_WAVE + lane / GL;  // row * groups + g
    const unsigned u = unit < units ? unit : units - 1, row = u / groups;
    float v[EL];
    load_el(v, x + (size_t)row * in_dim, (int)(u - row * groups) * GROUP + l * EL, in_dim, vec != 0);
    a8_oct(v, l, BITS, unit < units, xq + (size_t)u * GROUP, sx + u);
}

// R rows per workgroup, thread t holding positions 16 (t % (8 groups)) .. of
// row t / (8 groups).  The rows go to LDS once, for the chains: wavefront 0's
// lanes are R <= 4 rows x 16 accumulators, each reading its operand 16
// positions apart (rows 16 banks apart), a batch ahead of its fmas.  in_dim
// is a multiple of 16.
constexpr int NORM_R = 4;
constexpr int NORM_BATCH = 12;  // chain steps read at a time

template <int BITS>
__global__ __launch_bounds__(1024) void k_act_norm(const float* __restrict__ x, int rows, int in_dim, int groups,
                                                   int R, int vec, int vec_ns, const uint16_t* __restrict__ norm_scale,
                                                   int8_t* __restrict__ xq, float* __restrict__ sx) {
    extern __shared__ float xs[];  // [R][in_dim + 16]
    __shared__ float s_r[NORM_R];
    const int t = threadIdx.x, lane = t & 63, l = t & (GL - 1), pitch = in_dim + 16;
    const int rr = min(t / (GL * groups), R - 1), c = t - rr * GL * groups, p0 = c * EL, g = c / GL;
    const int row = (int)blockIdx.x * R + rr;
    const bool on = c < GL * groups && row < rows;
    const float* xr = x + (size_t)min(row, rows - 1) * in_dim;
    float v[EL];
    load_el(v, xr, p0, in_dim, vec != 0);
    // (16 positions at a time: in_dim and p0 are multiples of 16)
    const bool in = p0 < in_dim && c < GL * groups;
    uint32_t ns[EL / 2];
    {
        const uint16_t* sp = norm_scale + min(p0, in_dim - EL);
        if (vec_ns) {
            const uint4 a = reinterpret_cast<const uint4*>(sp)[0], b = reinterpret_cast<const uint4*>(sp)[1];
            ns[0] = a.x, ns[1] = a.y, ns[2] = a.z, ns[3] = a.w, ns[4] = b.x, ns[5] = b.y, ns[6] = b.z, ns[7] = b.w;
        } else {
#pragma unroll
            for (int i = 0; i < EL / 2; ++i) ns[i] = (uint32_t)sp[2 * i] | (uint32_t)sp[2 * i + 1] << 16;
        }
    }
    if (in) {
        float4* d = reinterpret_cast<float4*>(xs + rr * pitch + p0);
#pragma unroll
        for (int i = 0; i < EL / 4; ++i) d[i] = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
    }
    __syncthreads();
    if (t < 64) {
        // lane i16 = j * 4 + k of a row carries accumulator a[j][k] over
        // chunks ascending: a = fma(x[16 c + i16], x[16 c + i16], a)
        const int base = lane & 48, nc = in_dim / 16;
        const float* xc = xs + min(lane >> 4, R - 1) * pitch + (lane & 15);
        float a = 0.0f, buf[2][NORM_BATCH];
        auto fetch = [&](float (&b)[NORM_BATCH], int c0) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < NORM_BATCH; ++i) b[i] = xc[min(c0 + i, nc - 1) * 16];
        };
        auto chain = [&](const float (&b)[NORM_BATCH], int c0) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < NORM_BATCH; ++i)
                if (c0 + i < nc) a = __builtin_fmaf(b[i], b[i], a);
        };
        fetch(buf[0], 0);
        for (int c0 = 0; c0 < nc; c0 += 2 * NORM_BATCH) {
            fetch(buf[1], c0 + NORM_BATCH);
            __builtin_amdgcn_sched_barrier(0);
            chain(buf[0], c0);
            fetch(buf[0], c0 + 2 * NORM_BATCH);
            __builtin_amdgcn_sched_barrier(0);
            chain(buf[1], c0 + NORM_BATCH);
        }
        // t[k] = ((a[2][k] + a[3][k]) + a[1][k]) + a[0][k]
        const int k = base + (lane & 3);
        const float a0 = __shfl(a, k, 64), a1 = __shfl(a, k + 4, 64), a2 = __shfl(a, k + 8, 64),
                    a3 = __shfl(a, k + 12, 64);
        const float tk = ((a2 + a3) + a1) + a0;
        const float t0 = __shfl(tk, base, 64), t1 = __shfl(tk, base + 1, 64), t2 = __shfl(tk, base + 2, 64),
                    t3 = __shfl(tk, base + 3, 64);
        const float ss = (t0 + t1) + (t2 + t3);
        const float r = 1.0f / __builtin_sqrtf(ss / (float)in_dim + 1e-6f);
        if ((lane & 15) == 0) s_r[lane >> 4] = r;
    }
    __syncthreads();
    const float r = s_r[rr];
#pragma unroll
    for (int i = 0; i < EL; ++i) {
        const float tt = v[i] * r;
        v[i] = in ? __builtin_fmaf(tt, f16_bits_to_f32((uint16_t)(ns[i >> 1] >> (16 * (i & 1)))), tt) : 0.0f;
    }
    const size_t u = (size_t)min(row, rows - 1) * groups + min(g, groups - 1);
    a8_oct(v, l, BITS, on, xq + u * GROUP, sx + u);
}

hipError_t launch_act_prep(const float* x, int rows, int in_dim, int groups, int bits, const uint16_t* norm_scale,
                           int8_t* xq, float* sx, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    const int vec = (uintptr_t)x % 16 == 0 && in_dim % 4 == 0;
    if (!norm_scale) {
        const unsigned units = (unsigned)rows * (unsigned)groups;
        hipLaunchKernelGGL(bits == 2 ? k_act_a8<2> : k_act_a8<4>, dim3((units + ACT_WAVE - 1) / ACT_WAVE),
                           dim3(64), 0, s, x, units, in_dim,
                           (unsigned)groups, vec, xq, sx);
    } else {
        // up to four rows a workgroup within 512 threads and 64 KB of LDS
        const int R = std::min(std::min(rows, NORM_R), std::max(1, 512 / (GL * groups)));
        hipLaunchKernelGGL(bits == 2 ? k_act_norm<2> : k_act_norm<4>, dim3((rows + R - 1) / R),
                           dim3((R * GL * groups + 63) / 64 * 64), (size_t)R * (in_dim + 16) * 4, s, x, rows, in_dim,
                           groups, R, vec, (uintptr_t)norm_scale % 16 == 0, norm_scale, xq, sx);
    }
    return hipGetLastError();
}

}  // namespace nh
