// Row-wise block-128 Walsh-Hadamard with optional input/output scale vectors:
//   out[r, 128b + i] = (sum_j H[i, j] (in[r, 128b + j] * pre[128b + j])) * post[128b + i] * scale
// with H the Sylvester matrix / sqrt(128).  Replaces exllamav3_ext.had_r_128 as called at
// orcasaq2/ops.py:54 (pre = suh) and orcasaq2/ops.py:59 (post = svh, in place); the
// normalisation follows orcasaq2/__init__.py:39.  fp16 in/out, fp32 arithmetic.
//
// 16-byte-aligned pointers (the usual case): sixteen lanes per 128-block, four blocks per wave: lane l of a block holds elements
// 8(l % 16) .. 8(l % 16) + 7 (one 16-byte load and store).  Index bits 0..2 of the
// transform are inside a lane (three in-register butterfly stages), bits 3..6 are lane
// bits 0..3 (DPP exchanges inside each 16-lane row: quad_perm for 1 and 2, two banked
// row shifts for 4, row_ror:8 for 8).
#include "exl3_common.h"
#include "exl3_launch.h"

namespace exl3 {

constexpr int HAD_WAVES = 4;

// Words zero[0 .. nzero) to 0 by workgroup 0 (before any of its lanes leaves).
__device__ __forceinline__ void had_zero(uint32_t* zero, int nzero)
{
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < nzero; i += blockDim.x) zero[i] = 0u;
}

__global__ __launch_bounds__(64 * HAD_WAVES) void had_r_128_kernel(
    const uint4* in, uint4* out, const uint4* __restrict__ pre,  // in == out allowed
    const uint4* __restrict__ post, float scale, long blocks, int blocks_per_row, uint32_t* zero, int nzero, int in_bf, int out_bf, long ld_out)
{
    had_zero(zero, nzero);
    const long blk = ((long)blockIdx.x * HAD_WAVES + (threadIdx.x >> 6)) * 4 + ((threadIdx.x >> 4) & 3);
    if (blk >= blocks) return;  // no barriers or cross-row exchanges leave a 16-lane row
    const int lane = threadIdx.x & 15;
    const int col_blk = (int)(blk % blocks_per_row);
    float v[8];
    // loaded together: the conversion is behind a branch that would part the loads
    uint4 x = in[blk * 16 + lane], px = {0u, 0u, 0u, 0u}, qx = px;
    if (pre) px = pre[col_blk * 16 + lane];
    if (post) qx = post[col_blk * 16 + lane];
    if (in_bf) x = uint4{act_pair(x.x, 1), act_pair(x.y, 1), act_pair(x.z, 1), act_pair(x.w, 1)};
    had_unpack(x, v);
    if (pre) {
        float p[8];
        had_unpack(px, p);
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] *= p[i];
    }
    had16_stages(v, lane);
    float f[8];
#pragma unroll
    for (int i = 0; i < 8; i++) f[i] = 0.08838834764831845f * scale;   // 1/sqrt(128)
    if (post) {
        float p[8];
        had_unpack(qx, p);
#pragma unroll
        for (int i = 0; i < 8; i++) f[i] *= p[i];
    }
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] = out_pair(v[2 * i] * f[2 * i], v[2 * i + 1] * f[2 * i + 1], out_bf);
    out[(blk / blocks_per_row * ld_out + col_blk * 128) / 8 + lane] = uint4{o[0], o[1], o[2], o[3]};
}

// Pointers only 4-byte aligned: one wave per 128-block, lane l holds elements 2l, 2l + 1.
__global__ __launch_bounds__(64 * HAD_WAVES) void had_r_128_narrow_kernel(
    const uint32_t* in, uint32_t* out, const uint32_t* __restrict__ pre,  // in == out allowed
    const uint32_t* __restrict__ post, float scale, long blocks, int blocks_per_row, uint32_t* zero, int nzero, int in_bf, int out_bf, long ld_out)
{
    had_zero(zero, nzero);
    const long blk = (long)blockIdx.x * HAD_WAVES + (threadIdx.x >> 6);
    if (blk >= blocks) return;  // no barriers in this kernel
    const int lane = threadIdx.x & 63;
    const int col_blk = (int)(blk % blocks_per_row);
    const uint32_t v = act_pair(in[blk * 64 + lane], in_bf);
    float v0 = (float)__builtin_bit_cast(_Float16, (uint16_t)(v & 0xffffu));
    float v1 = (float)__builtin_bit_cast(_Float16, (uint16_t)(v >> 16));
    if (pre) {
        const uint32_t p = pre[col_blk * 64 + lane];
        v0 *= (float)__builtin_bit_cast(_Float16, (uint16_t)(p & 0xffffu));
        v1 *= (float)__builtin_bit_cast(_Float16, (uint16_t)(p >> 16));
    }
    wave_fwht128(v0, v1);
    if (post) {
        const uint32_t p = post[col_blk * 64 + lane];
        v0 *= (float)__builtin_bit_cast(_Float16, (uint16_t)(p & 0xffffu));
        v1 *= (float)__builtin_bit_cast(_Float16, (uint16_t)(p >> 16));
    }
    v0 *= scale;
    v1 *= scale;
    out[(blk / blocks_per_row * ld_out + col_blk * 128) / 2 + lane] = out_pair(v0, v1, out_bf);
}

int had_dispatch(const uint16_t* in, uint16_t* out, const uint16_t* pre, const uint16_t* post,
                 float scale, long rows, int cols, hipStream_t stream, uint32_t* zero, int nzero,
                 int in_bf, int out_bf, long ld_out)
{
    if (ld_out == 0) ld_out = cols;
    const int bpr = cols / 128;
    const long blocks = rows * bpr;
    if (blocks == 0 && nzero == 0) return EXL3_OK;   // with words to clear: one workgroup, no blocks
    auto a16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    if (!a16(in) || !a16(out) || ld_out % 8 || (pre && !a16(pre)) || (post && !a16(post))) {
        const long grid = std::max<long>(1, (blocks + HAD_WAVES - 1) / HAD_WAVES);
        hipLaunchKernelGGL(had_r_128_narrow_kernel, dim3((unsigned)grid), dim3(64 * HAD_WAVES), 0, stream,
                           reinterpret_cast<const uint32_t*>(in), reinterpret_cast<uint32_t*>(out),
                           reinterpret_cast<const uint32_t*>(pre), reinterpret_cast<const uint32_t*>(post),
                           scale, blocks, bpr, zero, nzero, in_bf, out_bf, ld_out);
        return check_launch("exl3_had_r_128");
    }
    const long grid = std::max<long>(1, (blocks + 4 * HAD_WAVES - 1) / (4 * HAD_WAVES));
    hipLaunchKernelGGL(had_r_128_kernel, dim3((unsigned)grid), dim3(64 * HAD_WAVES), 0, stream,
                       reinterpret_cast<const uint4*>(in), reinterpret_cast<uint4*>(out),
                       reinterpret_cast<const uint4*>(pre), reinterpret_cast<const uint4*>(post),
                       scale, blocks, bpr, zero, nzero, in_bf, out_bf, ld_out);
    return check_launch("exl3_had_r_128");
}

}  // namespace exl3
