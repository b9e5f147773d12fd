// LUT construction for gfx950 (MI355X): the one dense contraction of the path, on the matrix cores.
//
// Replaces model-calibration/pim_weight_converter.py:82-91 of the reference
//     lut = bmm(centroids.view(CB, C, v), weight.view(CB, v, M))
// and lut_quant (:21-35)
//     scale = max|lut| / 127;  q = int8(round_half_even(clamp(lut / scale, -128, 127))).
//
// One wave computes a 16-centroid x 64-column tile of one codebook with v_mfma_f32_16x16x4_f32
// (K = 4 matches sub_vec_len 4 in one step; other v loop/zero-pad).  The work is tiny
// (2*C*K*M flop) and the kernels are bound by reading W and writing the table once: the entries of an int8 table are computed twice, for
// their largest magnitude and again to be quantised, and never stored as floats -- a call needs a fifth of the device memory, and 768 ->
// 3072, 16 centroids takes 21 us of kernels instead of 29 (and 93 with a pass of its own over the table for the magnitudes).
#include "pimdl_internal.h"

namespace pimdl {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int LG_WAVES = 4;
constexpr int LG_FT = 4;  // 16-column tiles per wave
constexpr uint32_t LG_ORDERED = 8;  // centroids per thread of the ordered form

// largest value of a workgroup of four waves, in thread 0 (m >= 0; NaN is passed over)
__device__ __forceinline__ float block_max(float m)
{
    __shared__ float part[4];
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
    return fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
}

__device__ __forceinline__ int8_t quantise(float x, float scale)
{
    float t = __fdiv_rn(x, scale);
    t = fminf(fmaxf(t, -128.0f), 127.0f);
    return (int8_t)rintf(t);  // round half to even
}

// What a pass does with the entries that it computes
enum LutPass {
    LUT_STORE,     // float *out
    LUT_LARGEST,   // part [codebook][workgroups of a codebook]: the largest magnitude of each workgroup
    LUT_QUANTISE,  // int8 *out, with the scale of the codebook's group
};
struct LutOut {
    void* out;
    float* part;
    const float* scales;
    uint32_t group_cbs;  // codebooks per scale
};

// Lane (j, k) of a wave holds columns 4 j .. 4 j + 3 of its 64 (one per matrix instruction) of four centroids: whole 16-byte loads of W and
// 64 bytes of a table row per store and 16 lanes.
template <LutPass PASS>
__global__ __launch_bounds__(LG_WAVES * 64) void lutgen_kernel(const float* __restrict__ cent, const float* __restrict__ W, LutOut o,
                                                               uint32_t CB, uint32_t C, uint32_t v, uint32_t M)
{
    static_assert(LG_FT == 4, "four columns per lane");
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t j = lane & 15, k = lane >> 4;
    const uint32_t cb = blockIdx.z;
    const uint32_t c0 = blockIdx.y * 16;
    const uint32_t f0 = (blockIdx.x * LG_WAVES + wave) * (16 * LG_FT), f = f0 + 4 * j;
    const bool whole = M % 4 == 0;  // (uniform) else rows are not aligned to 16 bytes

    v4f acc[LG_FT];
#pragma unroll
    for (int t = 0; t < LG_FT; ++t) acc[t] = (v4f){0.f, 0.f, 0.f, 0.f};

    for (uint32_t t0 = 0; t0 < v && f0 < M; t0 += 4) {
        const uint32_t t = t0 + k;
        // A[i = centroid c0 + j][k = t]
        float a = 0.0f;
        if (c0 + j < C && t < v) a = cent[((size_t)cb * C + c0 + j) * v + t];
        v4f b = (v4f){0.f, 0.f, 0.f, 0.f};
        const float* w = W + ((size_t)cb * v + t) * M + f;
        if (whole) {
            if (t < v && f < M) b = *reinterpret_cast<const v4f*>(w);
        } else {
#pragma unroll
            for (int ft = 0; ft < LG_FT; ++ft)
                if (t < v && f + ft < M) b[ft] = w[ft];
        }
#pragma unroll
        for (int ft = 0; ft < LG_FT; ++ft) acc[ft] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b[ft], acc[ft], 0, 0, 0);
    }
    // D[i = 4*k + r][j]: centroid c0 + 4k + r, column f0 + 4 j + ft
    if constexpr (PASS == LUT_LARGEST) {
        // (rows past C and columns past M are sums of zeros)
        float m = 0.0f;
#pragma unroll
        for (int ft = 0; ft < LG_FT; ++ft)
#pragma unroll
            for (int r = 0; r < 4; ++r) m = fmaxf(m, fabsf(acc[ft][r]));
        m = block_max(m);
        if (threadIdx.x == 0) o.part[((size_t)cb * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x] = m;
    } else {
        const float scale = PASS == LUT_QUANTISE ? o.scales[cb / o.group_cbs] : 0.0f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t c = c0 + 4 * k + r;
            if (c >= C || f >= M) continue;
            const size_t at = ((size_t)cb * C + c) * M + f;
            if constexpr (PASS == LUT_STORE) {
                float* out = static_cast<float*>(o.out) + at;
                if (whole) *reinterpret_cast<v4f*>(out) = (v4f){acc[0][r], acc[1][r], acc[2][r], acc[3][r]};
                else
#pragma unroll
                    for (int ft = 0; ft < LG_FT; ++ft)
                        if (f + ft < M) out[ft] = acc[ft][r];
            } else {
                int8_t* out = static_cast<int8_t*>(o.out) + at;
                if (whole) *reinterpret_cast<char4*>(out) = make_char4(quantise(acc[0][r], scale), quantise(acc[1][r], scale), quantise(acc[2][r], scale), quantise(acc[3][r], scale));
                else
#pragma unroll
                    for (int ft = 0; ft < LG_FT; ++ft)
                        if (f + ft < M) out[ft] = quantise(acc[ft][r], scale);
            }
        }
    }
}

// The same product with the v terms of every entry added in ascending order, each multiplication and each
// addition rounded on its own, starting from 0.0f: the order in which a plain loop over the sub-vector runs
// on a CPU.  torch.bmm fixes no order (pim_weight_converter.py:86-90 leaves it to the library), so neither
// form is "the" reference result; this one makes a converter's output reproducible bit for bit by scalar code.
// One thread = one output column of one codebook, LG_ORDERED centroids one after the other: a small table is as long as this chain, and an int8
// one goes through it twice.  us a call, all centroids by one thread, from a table of floats that was kept / twice without it / by eights: 64 ->
// 64 v = 16, 64 centroids 142 / 206 / 65, v = 4 73 / 102 / 40; 256 -> 512 v = 16, 64 centroids 260 / 274 / 108; 768 -> 3072 v = 4, 16 centroids 637 / 545 / 522.
template <LutPass PASS>
__global__ __launch_bounds__(256) void lutgen_ordered_kernel(const float* __restrict__ cent, const float* __restrict__ W, LutOut o,
                                                           uint32_t C, uint32_t v, uint32_t M)
{
    const uint32_t groups = (C + LG_ORDERED - 1) / LG_ORDERED;  // workgroup x: centroid group x % groups of column tile x / groups
    const uint32_t f = blockIdx.x / groups * blockDim.x + threadIdx.x, cb = blockIdx.y, c0 = blockIdx.x % groups * LG_ORDERED;
    const uint32_t c1 = C - c0 < LG_ORDERED ? C : c0 + LG_ORDERED;
    const float* w = W + (size_t)cb * v * M + f;
    const float scale = PASS == LUT_QUANTISE ? o.scales[cb / o.group_cbs] : 0.0f;
    float m = 0.0f;
    for (uint32_t c = c0; c < c1 && f < M; ++c) {
        const float* a = cent + ((size_t)cb * C + c) * v;
        float acc = 0.0f;
        for (uint32_t t = 0; t < v; ++t) acc = __fadd_rn(acc, __fmul_rn(a[t], w[(size_t)t * M]));
        const size_t at = ((size_t)cb * C + c) * M + f;
        if constexpr (PASS == LUT_STORE) static_cast<float*>(o.out)[at] = acc;
        else if constexpr (PASS == LUT_QUANTISE) static_cast<int8_t*>(o.out)[at] = quantise(acc, scale);
        else m = fmaxf(m, fabsf(acc));
    }
    if constexpr (PASS == LUT_LARGEST) {
        m = block_max(m);
        if (threadIdx.x == 0) o.part[(size_t)cb * gridDim.x + blockIdx.x] = m;
    }
}

// A workgroup per group: its scale from the magnitudes of its codebooks' workgroups (parts per codebook).
__global__ __launch_bounds__(256) void lut_scale_kernel(const float* __restrict__ part, float* __restrict__ scales, uint32_t group_cbs,
                                                        uint32_t parts, uint32_t CB)
{
    const uint32_t grp = blockIdx.x, cb0 = grp * group_cbs, cb1 = CB - cb0 < group_cbs ? CB : cb0 + group_cbs;
    float m[8] = {};
    const uint64_t end = (uint64_t)cb1 * parts;
    for (uint64_t i = (uint64_t)cb0 * parts + threadIdx.x; i < end; i += 8 * 256)
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (i + 256 * u < end) m[u] = fmaxf(m[u], part[i + 256 * u]);
#pragma unroll
    for (int u = 1; u < 8; ++u) m[0] = fmaxf(m[0], m[u]);
    float scale = __fdiv_rn(block_max(m[0]), 127.0f);
    if (!(scale > 0.0f)) scale = 1.0f;  // all-zero group: any scale represents it
    if (threadIdx.x == 0) scales[grp] = scale;
}

// Pinned host memory to device memory or back (either side aligned to 16 bytes): the transfers of the ring in pimdl_capi.hip.  Four pieces of 16 bytes
// per thread are under way together, which the link's latency asks for.
__global__ __launch_bounds__(256) void ring_copy_kernel(const unsigned char* __restrict__ src, unsigned char* __restrict__ dst, uint64_t bytes)
{
    const uint4* s = reinterpret_cast<const uint4*>(src);
    uint4* d = reinterpret_cast<uint4*>(dst);
    const uint64_t n = bytes / 16, step = (uint64_t)gridDim.x * 256, first = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    for (uint64_t i = first; i < n; i += 4 * step) {
        uint4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (i + u * step < n) v[u] = s[i + u * step];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (i + u * step < n) d[i + u * step] = v[u];
    }
    for (uint64_t i = n * 16 + first; i < bytes; i += step) dst[i] = src[i];
}

// ---- diagnostics: a plain copy (HBM) and a ds_read_b128 loop (LDS) ------------------------------
__global__ void copy_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst, uint64_t n16)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (uint64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

typedef int v4i __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(1024) void lds_read_kernel(int* __restrict__ sink, int iters)
{
    __shared__ __attribute__((aligned(16))) int buf[16384];
    for (int i = threadIdx.x; i < 16384; i += blockDim.x) buf[i] = i;
    __syncthreads();
    const uint32_t addr = (threadIdx.x & 63) * 16;  // 64 lanes x 16 B: contiguous, conflict-free
    v4i s = {0, 0, 0, 0};
    for (int it = 0; it < iters; ++it) {
        v4i r0, r1, r2, r3, r4, r5, r6, r7;
        asm volatile(
            "ds_read_b128 %0, %8\n ds_read_b128 %1, %8 offset:4096\n ds_read_b128 %2, %8 offset:8192\n"
            "ds_read_b128 %3, %8 offset:12288\n ds_read_b128 %4, %8 offset:16384\n"
            "ds_read_b128 %5, %8 offset:20480\n ds_read_b128 %6, %8 offset:24576\n"
            "ds_read_b128 %7, %8 offset:28672\n s_waitcnt lgkmcnt(0)"
            : "=&v"(r0), "=&v"(r1), "=&v"(r2), "=&v"(r3), "=&v"(r4), "=&v"(r5), "=&v"(r6), "=&v"(r7)
            : "v"(addr));
        s += r0 + r1 + r2 + r3 + r4 + r5 + r6 + r7;
    }
    sink[blockIdx.x * blockDim.x + threadIdx.x] = s.x + s.y + s.z + s.w;
}

}  // namespace

// workgroups per codebook, each of which leaves its largest magnitude
uint32_t lutgen_parts(uint32_t C, uint32_t M, bool ordered)
{
    return ordered ? (M + 255) / 256 * ((C + LG_ORDERED - 1) / LG_ORDERED) : (M + LG_WAVES * 16 * LG_FT - 1) / (LG_WAVES * 16 * LG_FT) * ((C + 15) / 16);
}

template <LutPass PASS>
static int launch_pass(Ctx* ctx, const float* d_cent, const float* d_w, const LutOut& o, uint32_t CB, uint32_t C, uint32_t v, uint32_t M, bool ordered)
{
    if (ordered) {
        hipLaunchKernelGGL(lutgen_ordered_kernel<PASS>, dim3(lutgen_parts(C, M, true), CB), dim3(256), 0, ctx->stream, d_cent, d_w, o, C, v, M);
        return hip_check(ctx, hipGetLastError(), "lutgen_ordered_kernel launch");
    }
    dim3 grid((M + LG_WAVES * 16 * LG_FT - 1) / (LG_WAVES * 16 * LG_FT), (C + 15) / 16, CB);
    hipLaunchKernelGGL(lutgen_kernel<PASS>, grid, dim3(LG_WAVES * 64), 0, ctx->stream, d_cent, d_w, o, CB, C, v, M);
    return hip_check(ctx, hipGetLastError(), "lutgen_kernel launch");
}

int launch_lutgen_f32(Ctx* ctx, const float* d_cent, const float* d_w, float* d_lut, uint32_t CB, uint32_t C, uint32_t v, uint32_t M, bool ordered)
{
    return launch_pass<LUT_STORE>(ctx, d_cent, d_w, LutOut{d_lut, nullptr, nullptr, 1}, CB, C, v, M, ordered);
}

int launch_lutgen_i8(Ctx* ctx, const float* d_cent, const float* d_w, float* d_part, int8_t* d_q, float* d_scales, uint32_t CB, uint32_t C,
                     uint32_t v, uint32_t M, uint32_t scale_group, bool ordered)
{
    const uint32_t cbs = scale_group && scale_group < CB ? scale_group : CB, ngroups = (CB + cbs - 1) / cbs;
    const LutOut o{d_q, d_part, d_scales, cbs};
    int rc = launch_pass<LUT_LARGEST>(ctx, d_cent, d_w, o, CB, C, v, M, ordered);
    if (rc) return rc;
    hipLaunchKernelGGL(lut_scale_kernel, dim3(ngroups), dim3(256), 0, ctx->stream, d_part, d_scales, cbs, lutgen_parts(C, M, ordered), CB);
    if ((rc = hip_check(ctx, hipGetLastError(), "lut_scale_kernel launch"))) return rc;
    return launch_pass<LUT_QUANTISE>(ctx, d_cent, d_w, o, CB, C, v, M, ordered);
}

int launch_ring_copy(Ctx* ctx, const void* src, void* dst, size_t bytes)
{
    const uint64_t wgs = (bytes + 256 * 64 - 1) / (256 * 64);
    hipLaunchKernelGGL(ring_copy_kernel, dim3((uint32_t)(wgs < 128 ? wgs : 128)), dim3(256), 0, ctx->stream, static_cast<const unsigned char*>(src),
                       static_cast<unsigned char*>(dst), (uint64_t)bytes);
    return hip_check(ctx, hipGetLastError(), "ring_copy_kernel launch");
}

int launch_diag(Ctx* ctx, uint64_t bytes, float* copy_gbps, float* lds_gbps)
{
    int rc = PIMDL_OK;
    if (copy_gbps) {
        const uint64_t n16 = bytes / 16;
        if (n16 == 0) return set_error(ctx, PIMDL_ERR_INVALID, "pimdl_diag_bandwidth: bytes < 16");
        uint4 *src = nullptr, *dst = nullptr;
        if ((rc = hip_check(ctx, hipMalloc(&src, n16 * 16), "hipMalloc(diag src)"))) return rc;
        if ((rc = hip_check(ctx, hipMalloc(&dst, n16 * 16), "hipMalloc(diag dst)"))) { (void)hipFree(src); return rc; }
        (void)hipMemsetAsync(src, 1, n16 * 16, ctx->stream);
        const uint32_t blocks = ctx->prop.multiProcessorCount * 8;
        for (int w = 0; w < 2; ++w) hipLaunchKernelGGL(copy_kernel, dim3(blocks), dim3(256), 0, ctx->stream, src, dst, n16);
        (void)hipEventRecord(ctx->ev[0], ctx->stream);
        const int reps = 10;
        for (int w = 0; w < reps; ++w) hipLaunchKernelGGL(copy_kernel, dim3(blocks), dim3(256), 0, ctx->stream, src, dst, n16);
        (void)hipEventRecord(ctx->ev[1], ctx->stream);
        rc = hip_check(ctx, hipEventSynchronize(ctx->ev[1]), "diag copy");
        float ms = 0;
        (void)hipEventElapsedTime(&ms, ctx->ev[0], ctx->ev[1]);
        *copy_gbps = ms > 0 ? (float)(2.0 * n16 * 16 * reps / (ms * 1e6)) : 0.f;  // read + write
        (void)hipFree(src);
        (void)hipFree(dst);
        if (rc) return rc;
    }
    if (lds_gbps) {
        const uint32_t blocks = ctx->prop.multiProcessorCount * 2, threads = 1024;
        int* sink = nullptr;
        if ((rc = hip_check(ctx, hipMalloc(&sink, (size_t)blocks * threads * 4), "hipMalloc(diag sink)"))) return rc;
        const int iters = 4000;
        hipLaunchKernelGGL(lds_read_kernel, dim3(blocks), dim3(threads), 0, ctx->stream, sink, iters);
        (void)hipEventRecord(ctx->ev[0], ctx->stream);
        hipLaunchKernelGGL(lds_read_kernel, dim3(blocks), dim3(threads), 0, ctx->stream, sink, iters);
        (void)hipEventRecord(ctx->ev[1], ctx->stream);
        rc = hip_check(ctx, hipEventSynchronize(ctx->ev[1]), "diag lds");
        float ms = 0;
        (void)hipEventElapsedTime(&ms, ctx->ev[0], ctx->ev[1]);
        *lds_gbps = ms > 0 ? (float)((double)blocks * threads * iters * 8 * 16 / (ms * 1e6)) : 0.f;
        (void)hipFree(sink);
    }
    return rc;
}

}  // namespace pimdl
