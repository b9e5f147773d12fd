// Layer normalisation of the reference's transformer layer for gfx950 (MI355X).
//
// Replaces norm() (inference-engine/src/host/transformer_layer.cpp:50-90) and the residual add that
// follows it in the layer (:476-486 and :601-611).  Numerics follow the reference statement by
// statement: the mean and the variance are accumulated in double and rounded to float, the centred
// value, its square and the three output operations (scale, weight, bias) are separately rounded fp32
// operations (this translation unit is built with -ffp-contract=off), eps = 1e-6.  The only freedom
// taken is the order of the two double-precision sums: a row is summed by 64 lanes and a butterfly
// instead of sequentially, which can move the float mean or variance by one ulp in rare rows.
// The centred value x - mean is computed once and reused (the reference computes the identical
// expression twice).
#include <type_traits>

#include "pimdl_internal.h"

namespace pimdl {

namespace {

// The value of lane ^ OFF (for OFF < 8: of a lane that holds the same value, given that the steps above were done before,
// which leave values that repeat every 2 * OFF lanes), without the LDS crossbar's round trip: half-wave and row swaps, then
// rotations within a row of 16 and a quad.
template <int OFF>
__device__ __forceinline__ void xor_pair(uint32_t v, uint32_t& a, uint32_t& b)
{
    if constexpr (OFF >= 16) {  // a: the lower halves (rows) in both places, b: the upper ones
        auto r = [&] {
            if constexpr (OFF == 32) return __builtin_amdgcn_permlane32_swap(v, v, false, false);
            else return __builtin_amdgcn_permlane16_swap(v, v, false, false);
        }();
        a = r[0];
        b = r[1];
    } else {
        constexpr int ctrl = OFF == 8 ? 0x128 : OFF == 4 ? 0x124 : OFF == 2 ? 0x4E : 0xB1;  // row_ror:8, row_ror:4, quad_perm
        a = v;
        b = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, 0xF, 0xF, true);
    }
}

template <int OFF>
__device__ __forceinline__ double add_pair(double v)
{
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    uint32_t alo, blo, ahi, bhi;
    xor_pair<OFF>((uint32_t)u, alo, blo);
    xor_pair<OFF>((uint32_t)(u >> 32), ahi, bhi);
    return __longlong_as_double((long long)((uint64_t)ahi << 32 | alo)) + __longlong_as_double((long long)((uint64_t)bhi << 32 | blo));
}

// Butterfly over the 64 lanes, 32 lanes apart first: the same additions, and so the same bits, as with __shfl_xor, whose
// twelve trips through the LDS crossbar per sum stood in the wave's only chain (us in a layer: d = 768, n = 4096
// 8.1 -> 7.65, with the registers of a row cut to its 768 columns; d = 1024, n = 8192 17.5 -> 16.8).
__device__ __forceinline__ double wave_sum(double v)
{
    v = add_pair<32>(v);
    v = add_pair<16>(v);
    v = add_pair<8>(v);
    v = add_pair<4>(v);
    v = add_pair<2>(v);
    return add_pair<1>(v);
}

// one wave per row
__global__ __launch_bounds__(256) void layer_norm_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                        const float* __restrict__ b,
                                                        const float* __restrict__ residual,
                                                        float* __restrict__ out, uint32_t n, uint32_t d, float eps)
{
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= n) return;
    const float* xr = x + (size_t)row * d;
    double s = 0.0;
    for (uint32_t i = lane; i < d; i += 64) s += (double)xr[i];
    const float mean = (float)(wave_sum(s) / (double)d);
    double s2 = 0.0;
    for (uint32_t i = lane; i < d; i += 64) {
        const float v = __fsub_rn(xr[i], mean);
        s2 += (double)__fmul_rn(v, v);
    }
    const float variance = (float)(wave_sum(s2) / (double)d);
    const float scale = 1.0f / sqrtf(__fadd_rn(variance, eps));
    float* o = out + (size_t)row * d;
    const float* r = residual ? residual + (size_t)row * d : nullptr;
    for (uint32_t i = lane; i < d; i += 64) {
        float y = __fsub_rn(xr[i], mean);
        y = __fmul_rn(y, scale);
        y = __fmul_rn(y, w[i]);
        y = __fadd_rn(y, b[i]);
        o[i] = r ? __fadd_rn(r[i], y) : y;
    }
}

// The same for rows of up to 64 * 4 * KV floats with d % 4 == 0 and 16-byte aligned buffers: the row
// is read once with float4 loads and stays in registers for the three passes.  Weight, bias and residual are
// requested together with the row, ahead of the two reductions, so that the wave waits for memory once.
template <int KV>
__global__ __launch_bounds__(256) void layer_norm_vec_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                            const float* __restrict__ b,
                                                            const float* __restrict__ residual,
                                                            float* __restrict__ out, uint32_t n, uint32_t d, float eps)
{
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= n) return;
    const uint32_t d4 = d / 4;
    const float4* xr = reinterpret_cast<const float4*>(x + (size_t)row * d);
    float4 xv[KV], wv[KV], bv[KV], rv[KV];
    const float4* r = residual ? reinterpret_cast<const float4*>(residual + (size_t)row * d) : nullptr;
    const float4* w4 = reinterpret_cast<const float4*>(w);
    const float4* b4 = reinterpret_cast<const float4*>(b);
#pragma unroll
    for (int k = 0; k < KV; ++k) {
        const uint32_t i = lane + 64 * k;
        if (i < d4) {
            xv[k] = xr[i];
            wv[k] = w4[i];
            bv[k] = b4[i];
            if (r) rv[k] = r[i];
        }
    }
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < KV; ++k) {
        const uint32_t i = lane + 64 * k;
        if (i < d4) {
            s += (double)xv[k].x;
            s += (double)xv[k].y;
            s += (double)xv[k].z;
            s += (double)xv[k].w;
        }
    }
    const float mean = (float)(wave_sum(s) / (double)d);
    double s2 = 0.0;
#pragma unroll
    for (int k = 0; k < KV; ++k) {
        if (lane + 64 * k < d4) {
            xv[k].x = __fsub_rn(xv[k].x, mean);
            xv[k].y = __fsub_rn(xv[k].y, mean);
            xv[k].z = __fsub_rn(xv[k].z, mean);
            xv[k].w = __fsub_rn(xv[k].w, mean);
            s2 += (double)__fmul_rn(xv[k].x, xv[k].x);
            s2 += (double)__fmul_rn(xv[k].y, xv[k].y);
            s2 += (double)__fmul_rn(xv[k].z, xv[k].z);
            s2 += (double)__fmul_rn(xv[k].w, xv[k].w);
        }
    }
    const float variance = (float)(wave_sum(s2) / (double)d);
    const float scale = 1.0f / sqrtf(__fadd_rn(variance, eps));
    float4* o = reinterpret_cast<float4*>(out + (size_t)row * d);
#pragma unroll
    for (int k = 0; k < KV; ++k) {
        const uint32_t i = lane + 64 * k;
        if (i < d4) {
            float4 y;
            y.x = __fadd_rn(__fmul_rn(__fmul_rn(xv[k].x, scale), wv[k].x), bv[k].x);
            y.y = __fadd_rn(__fmul_rn(__fmul_rn(xv[k].y, scale), wv[k].y), bv[k].y);
            y.z = __fadd_rn(__fmul_rn(__fmul_rn(xv[k].z, scale), wv[k].z), bv[k].z);
            y.w = __fadd_rn(__fmul_rn(__fmul_rn(xv[k].w, scale), wv[k].w), bv[k].w);
            if (r) {
                y.x = __fadd_rn(rv[k].x, y.x);
                y.y = __fadd_rn(rv[k].y, y.y);
                y.z = __fadd_rn(rv[k].z, y.z);
                y.w = __fadd_rn(rv[k].w, y.w);
            }
            o[i] = y;
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Unmasked multi-head attention, softmax(q k^T * scale) v per (batch, head), fp32, head_dim 64.
// Replaces the attention step of the reference's layer (src/host/transformer_layer.cpp:211-230:
// KQ = K Q, scale by 1/sqrt(head_dim), soft_max, V KQ, permute back to [n][token_dim]); inputs and
// output stay in the layer's [token][head * 64 + d] order, so no head transposes are needed.
//
// A workgroup = 64 queries of one (batch, head), a wave = 16 of them.  Keys are taken in chunks of 128, with the running
// maximum / sum of a streaming softmax between chunks.  A chunk's K and then its V go through LDS in pieces of 32 keys, copied without
// registers (global_load_lds) into a ring of four: when a piece is worked on, the next two have been requested and the
// third goes into the place of the piece before, so there is one barrier per piece and the first products wait for 32 keys, not
// for 128.  Key tiles of 16 past the end of the sequence are skipped.  Both products run on v_mfma_f32_16x16x4_f32,
// transposed so that nothing has to change lanes in between:
//   S^T[key][query]  = K Q^T:  A = K rows (keys), B = this lane's query, 16 steps of 4 dims.  The K
//                      index of lane group g in step s is dim 16 g + s (a sum does not care in which
//                      order its terms are paired), so a lane's operands are 16 consecutive floats.
//                      Result: lane (query j, group g) holds keys 16 kt + 4 g + i of key tile kt.
//   out^T[d][query] += V^T P^T: the B operand of step (kt, i) is that very register (key 16 kt + 4 g + i
//                      from group g), A = V[that key][16 dt + j].  Result: lane (j, g) holds dims
//                      16 dt + 4 g + i of its query: one float4 store per 16-dim tile.
// A row of a piece is 64 floats, all LDS banks once.  Rows lie in fours, 64 bytes between one four and the next, and the 16-byte
// parts of a row in the order part ^ (row % 4): so the 16 dims x 4 keys of the second product's reads fall into different banks, and
// everything but the lane's own place is an immediate offset of the read.  Of the first product's reads (16 keys x 4 groups, served 16
// lanes at a time) two lanes meet in a bank, 4 cycles more for each: a quarter of the LDS's cycles, which are 15 to 17 % of the kernel's.
// What bounds it: the fp32 matrix instructions and the vector ones share a unit, so the kernel takes the sum of their
// times; everything that a whole chunk does not need (masks, clamped rows, zeroed rows) is compiled for the last chunk alone.
// us, before (whole chunks through registers, four barriers each, masks in every chunk, three workgroups per CU) / now, same bits:
// 32 x 128 tokens, 12 heads 24.6 / 21.4; 64 x 128, 16 heads 51.9 / 46; 64 x 197, 12 heads 112 / 102; 16 x 512, 12 heads 131 / 115 (82 of
// them matrix instructions at 2.4 GHz); 300 x 17, 12 heads 33 / 27; 1 x 128, 12 heads 9.9 / 8.2.  (The ring alone, with the masks and
// clamped addresses left in every chunk: 24.5, 51.3, 112.8, 129, 41, 10.2 -- it is the vector instructions that count.)
// ---------------------------------------------------------------------------------------------
constexpr int AT_KC = 128, AT_PK = 32, AT_PIECES = AT_KC / AT_PK, AT_THREADS = 256;
constexpr int AT_FOUR = 4 * 256 + 64, AT_TILE = 4 * AT_FOUR, AT_PIECE_BYTES = 2 * AT_TILE;  // bytes of 4, 16 and 32 rows
typedef float v4f __attribute__((ext_vector_type(4)));

template <int OFF>
__device__ __forceinline__ void at_read(v4f& dst, uint32_t addr)
{
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}
template <int OFF>
__device__ __forceinline__ void at_read(float& dst, uint32_t addr)
{
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}
template <int N>
__device__ __forceinline__ void at_lgkm_wait()
{
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory");
    __builtin_amdgcn_sched_barrier(0);
}

__global__ __launch_bounds__(AT_THREADS, 4) void attention_hd64_kernel(const float* __restrict__ q,
                                                                   const float* __restrict__ k,
                                                                   const float* __restrict__ v,
                                                                   float* __restrict__ out, uint32_t S,
                                                                   uint32_t in_stride, uint32_t out_stride,
                                                                   float scale)
{
    __shared__ __attribute__((aligned(1024))) unsigned char kv[AT_PIECES * AT_PIECE_BYTES];
    const uint32_t h = blockIdx.y, b = blockIdx.z;
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t j = lane & 15, g = lane >> 4;
    const size_t in_base = (size_t)b * S * in_stride + (size_t)h * 64;
    const uint32_t q_tok = blockIdx.x * 64 + wave * 16 + j;
    const uint32_t q_tok_c = q_tok < S ? q_tok : S - 1;  // rows past S repeat the last query; never stored

    v4f qraw[4];
    {
        const float* qp = q + in_base + (size_t)q_tok_c * in_stride + 16 * g;
#pragma unroll
        for (int i = 0; i < 4; ++i) qraw[i] = *reinterpret_cast<const v4f*>(qp + 4 * i);
    }
    // Copies this wave's 8 rows of a piece (two operations of 4 rows).  CLAMP: rows past the sequence repeat its last one.
    const uint32_t part = (j & 12) | ((j & 3) ^ g);  // that this lane copies of its row
    const size_t copy_off[2] = {((size_t)(wave * 8 + g) * in_stride + 4 * part) * 4, ((size_t)(wave * 8 + 4 + g) * in_stride + 4 * part) * 4};
    auto copy_piece = [&](const float* src, uint32_t key0, auto slotc, auto clampc) __attribute__((always_inline)) {
        constexpr int slot = decltype(slotc)::value;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const char* p;
            if constexpr (decltype(clampc)::value) {
                const uint32_t key = key0 + wave * 8 + 4 * u + g, tok = key < S ? key : S - 1;
                p = reinterpret_cast<const char*>(src + in_base + (size_t)tok * in_stride + 4 * part);
            } else {
                p = reinterpret_cast<const char*>(src + in_base + (size_t)key0 * in_stride) + copy_off[u];
            }
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)p,
                                             (__attribute__((address_space(3))) void*)(kv + slot * AT_PIECE_BYTES + (2 * wave + u) * AT_FOUR), 16, 0, 0);
        }
    };
    // The piece about to be used has landed (`behind` operations have been issued since), then everybody's part of it; after
    // that everybody is done with the piece before.
    auto arrive = [&](auto behindc) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(behindc)::value) : "memory");
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)kv);
    // K rows: part 4 g + i of row j; V: float j % 4 of part 4 dt + j / 4 of row 4 g + i
    uint32_t k_addr[4], v_addr[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        k_addr[i] = lds0 + j / 4 * AT_FOUR + j % 4 * 256 + (4 * g + (i ^ (j & 3))) * 16;
        v_addr[i] = lds0 + g * AT_FOUR + i * 256 + ((j / 4) ^ i) * 16 + (j % 4) * 4;
    }

    constexpr std::integral_constant<int, 0> c0;
    constexpr std::integral_constant<int, 1> c1;
    constexpr std::integral_constant<int, 2> c2;
    constexpr std::integral_constant<int, 3> c3;
    // The three pieces that the chunk at kc begins with: of K -- or, where at most 64 keys are left (short chunk), K, K and V,
    // whose places are 2 and 3 then.
    auto begin_piece = [&](uint32_t kc, auto pc) __attribute__((always_inline)) {
        constexpr int p = decltype(pc)::value;
        if (kc + AT_KC <= S) copy_piece(k, kc + p * AT_PK, pc, std::false_type{});
        else if (p < 2 || kc + 2 * AT_PK < S) copy_piece(k, kc + p * AT_PK, pc, std::true_type{});
        else copy_piece(v, kc, pc, std::true_type{});
    };
    begin_piece(0, c0);
    begin_piece(0, c1);
    begin_piece(0, c2);
    float qreg[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) qreg[i] = qraw[i / 4][i % 4] * scale;

    float m_run = -__builtin_inff(), l_run = 0.0f;
    v4f o[4];
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) o[dt] = (v4f){0.f, 0.f, 0.f, 0.f};

    // WHOLE: 128 keys, SHORT: at most 64; LAST: no chunk follows
    auto chunk = [&](uint32_t kc, auto wholec, auto shortc, auto lastc) __attribute__((always_inline)) {
        constexpr bool WHOLE = decltype(wholec)::value, SHORT = decltype(shortc)::value, LAST = decltype(lastc)::value;
        constexpr std::bool_constant<!WHOLE> tail;
        constexpr int TILES = SHORT ? 4 : AT_KC / 16, V0 = SHORT ? 2 : 0;  // key tiles; place of the first piece of V
        const bool two = kc + AT_PK < S;  // (SHORT) pieces
        v4f s[TILES];
        auto scores = [&](auto pc) __attribute__((always_inline)) {
            constexpr int p = decltype(pc)::value;
            v4f a[2][4];
            auto request = [&](auto tc) {
                constexpr int t = decltype(tc)::value, off = p * AT_PIECE_BYTES + t * AT_TILE;
                at_read<off>(a[t][0], k_addr[0]);
                at_read<off>(a[t][1], k_addr[1]);
                at_read<off>(a[t][2], k_addr[2]);
                at_read<off>(a[t][3], k_addr[3]);
            };
            auto product = [&](auto tc) {
                constexpr int t = decltype(tc)::value, kt = 2 * p + t;
#pragma unroll
                for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(a[t][i]));
                s[kt] = (v4f){0.f, 0.f, 0.f, 0.f};
                if (WHOLE || kc + 16 * kt < S) {  // (uniform) else a key tile past the sequence: nothing to compute
#pragma unroll
                    for (int st = 0; st < 16; ++st) s[kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t][st / 4][st % 4], qreg[st], s[kt], 0, 0, 0);
                }
            };
            request(c0);
            request(c1);
            at_lgkm_wait<4>();
            product(c0);
            at_lgkm_wait<0>();
            product(c1);
        };
        arrive(std::integral_constant<int, 4>{});
        if constexpr (SHORT) {
            if (two) copy_piece(v, kc + AT_PK, c3, tail);
            scores(c0);
            if (two) {
                arrive(std::integral_constant<int, 4>{});
                scores(c1);
            } else {
                s[2] = s[3] = (v4f){0.f, 0.f, 0.f, 0.f};
            }
        } else {
            copy_piece(k, kc + 3 * AT_PK, c3, tail);
            scores(c0);
            arrive(std::integral_constant<int, 4>{});
            copy_piece(v, kc, c0, tail);
            scores(c1);
            arrive(std::integral_constant<int, 4>{});
            copy_piece(v, kc + AT_PK, c1, tail);
            scores(c2);
            arrive(std::integral_constant<int, 4>{});
            copy_piece(v, kc + 2 * AT_PK, c2, tail);
            scores(c3);
        }

        // keys past S do not take part
        float mx = -__builtin_inff();
#pragma unroll
        for (int kt = 0; kt < TILES; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (!WHOLE && kc + 16 * kt + 4 * g + i >= S) s[kt][i] = -__builtin_inff();
                mx = fmaxf(mx, s[kt][i]);
            }
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float m_new = fmaxf(m_run, mx);  // finite: key kc exists
        const float alpha = __expf(m_run - m_new);  // 0 for the first chunk
        float psum = 0.0f;
#pragma unroll
        for (int kt = 0; kt < TILES; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float p = __expf(s[kt][i] - m_new);
                s[kt][i] = p;
                psum += p;
            }
        psum += __shfl_xor(psum, 16);
        psum += __shfl_xor(psum, 32);
        l_run = l_run * alpha + psum;
        m_run = m_new;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) o[dt] *= alpha;

        // rows of V past the sequence must be zeros (their probabilities are, but zero times infinity is not)
        auto zero_rows = [&](auto pc) {
            constexpr int p = decltype(pc)::value;
            const uint32_t key0 = kc + p * AT_PK;
            if (WHOLE || key0 + AT_PK <= S || key0 >= S) return;  // (uniform)
#pragma unroll
            for (int u = 0; u < 2; ++u)
                if (key0 + wave * 8 + 4 * u + g >= S)
                    *reinterpret_cast<v4f*>(kv + (V0 + p) * AT_PIECE_BYTES + (2 * wave + u) * AT_FOUR + lane * 16) = (v4f){0.f, 0.f, 0.f, 0.f};
        };
        auto values = [&](auto pc) __attribute__((always_inline)) {
            constexpr int p = decltype(pc)::value;
            float a[4][4];
            auto request = [&](auto tc, auto ic) {
                constexpr int off = (V0 + p) * AT_PIECE_BYTES + decltype(tc)::value * AT_TILE, i = decltype(ic)::value;
                at_read<off>(a[i][0], v_addr[i]);
                at_read<off + 64>(a[i][1], v_addr[i]);
                at_read<off + 128>(a[i][2], v_addr[i]);
                at_read<off + 192>(a[i][3], v_addr[i]);
            };
            auto product = [&](auto tc, auto ic) {
                constexpr int kt = 2 * p + decltype(tc)::value, i = decltype(ic)::value;
#pragma unroll
                for (int dt = 0; dt < 4; ++dt) asm volatile("" : "+v"(a[i][dt]));
                if (WHOLE || kc + 16 * kt < S) {  // (uniform) else its probabilities are all zero
#pragma unroll
                    for (int dt = 0; dt < 4; ++dt) o[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][dt], s[kt][i], o[dt], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            request(c0, c0);
            request(c0, c1);
            request(c0, c2);
            request(c0, c3);
            at_lgkm_wait<12>();
            product(c0, c0);
            request(c1, c0);
            at_lgkm_wait<12>();
            product(c0, c1);
            request(c1, c1);
            at_lgkm_wait<12>();
            product(c0, c2);
            request(c1, c2);
            at_lgkm_wait<12>();
            product(c0, c3);
            request(c1, c3);
            at_lgkm_wait<12>();
            product(c1, c0);
            at_lgkm_wait<8>();
            product(c1, c1);
            at_lgkm_wait<4>();
            product(c1, c2);
            at_lgkm_wait<0>();
            product(c1, c3);
        };
        auto arrive_v = [&](auto pc, auto behindc) {  // (behindc: where no chunk follows)
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LAST ? decltype(behindc)::value : 4) : "memory");
            zero_rows(pc);
            __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
        };
        auto next_piece = [&](auto pc) {
            if constexpr (!LAST) begin_piece(kc + AT_KC, pc);
        };
        if constexpr (SHORT) {
            if (two) {
                arrive_v(c0, std::integral_constant<int, 2>{});
                values(c0);
                arrive_v(c1, std::integral_constant<int, 0>{});
                values(c1);
            } else {
                arrive_v(c0, std::integral_constant<int, 0>{});
                values(c0);
            }
        } else {
            arrive_v(c0, std::integral_constant<int, 4>{});
            copy_piece(v, kc + 3 * AT_PK, c3, tail);
            values(c0);
            arrive_v(c1, std::integral_constant<int, 4>{});
            next_piece(c0);
            values(c1);
            arrive_v(c2, std::integral_constant<int, 2>{});
            next_piece(c1);
            values(c2);
            arrive_v(c3, std::integral_constant<int, 0>{});
            next_piece(c2);
            values(c3);
        }
    };
    constexpr std::true_type yes;
    constexpr std::false_type no;
    uint32_t kc = 0;
    for (; kc + AT_KC < S; kc += AT_KC) chunk(kc, yes, no, no);
    if (kc + AT_KC == S) chunk(kc, yes, no, yes);
    else if (kc + 2 * AT_PK < S) chunk(kc, no, no, yes);
    else chunk(kc, no, yes, yes);
    if (q_tok < S) {
        const float inv = 1.0f / l_run;
        float* op = out + ((size_t)b * S + q_tok) * out_stride + (size_t)h * 64 + 4 * g;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
            *reinterpret_cast<float4*>(op + 16 * dt) = make_float4(o[dt][0] * inv, o[dt][1] * inv, o[dt][2] * inv, o[dt][3] * inv);
    }
}

}  // namespace

// Shapes are checked by the caller (head_dim 64, strides multiples of 4 floats, 16-byte aligned pointers).
int launch_attention_hd64(Ctx* ctx, const float* d_q, const float* d_k, const float* d_v, float* d_out, uint32_t batch,
                          uint32_t seq, uint32_t heads, uint32_t in_stride, uint32_t out_stride, float scale)
{
    if (batch == 0 || seq == 0 || heads == 0) return PIMDL_OK;
    hipLaunchKernelGGL(attention_hd64_kernel, dim3((seq + 63) / 64, heads, batch), dim3(AT_THREADS), 0, ctx->stream, d_q,
                       d_k, d_v, d_out, seq, in_stride, out_stride, scale);
    return hip_check(ctx, hipGetLastError(), "attention_hd64_kernel launch");
}

int launch_layer_norm(Ctx* ctx, const float* d_x, const float* d_w, const float* d_b, const float* d_residual,
                      float* d_out, uint32_t n, uint32_t d, float eps)
{
    if (n == 0) return PIMDL_OK;
    const uintptr_t all = reinterpret_cast<uintptr_t>(d_x) | reinterpret_cast<uintptr_t>(d_w) |
                          reinterpret_cast<uintptr_t>(d_b) | reinterpret_cast<uintptr_t>(d_residual) |
                          reinterpret_cast<uintptr_t>(d_out);
    if (d % 4 == 0 && (all & 15) == 0 && d <= 64 * 4 * 8) {
        if (d <= 64 * 4 * 3)
            hipLaunchKernelGGL(layer_norm_vec_kernel<3>, dim3((n + 3) / 4), dim3(256), 0, ctx->stream, d_x, d_w, d_b,
                               d_residual, d_out, n, d, eps);
        else if (d <= 64 * 4 * 4)
            hipLaunchKernelGGL(layer_norm_vec_kernel<4>, dim3((n + 3) / 4), dim3(256), 0, ctx->stream, d_x, d_w, d_b,
                               d_residual, d_out, n, d, eps);
        else
            hipLaunchKernelGGL(layer_norm_vec_kernel<8>, dim3((n + 3) / 4), dim3(256), 0, ctx->stream, d_x, d_w, d_b,
                               d_residual, d_out, n, d, eps);
        return hip_check(ctx, hipGetLastError(), "layer_norm_vec_kernel launch");
    }
    hipLaunchKernelGGL(layer_norm_kernel, dim3((n + 3) / 4), dim3(256), 0, ctx->stream, d_x, d_w, d_b, d_residual,
                       d_out, n, d, eps);
    return hip_check(ctx, hipGetLastError(), "layer_norm_kernel launch");
}

}  // namespace pimdl
