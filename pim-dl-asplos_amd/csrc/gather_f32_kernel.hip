// LUT gather-accumulate for tables resident as floats with up to 32 centroids (gfx950): fp32 tables, and int8 tables with a
// scale per group of codebooks.
//     out[n][f] = (sum over cb ascending, fp32) lut[cb][idx[n][cb]][f] + bias[f]
// (inference-engine/test/test_amm.cpp:164-175 on a float table).  The order of the additions is part of the result, so
// every gathered entry costs one read from LDS and one vector addition, whatever the kernel: N * CB * M additions at 16
// lanes per clock and SIMD, and 4 * N * CB * M bytes at 256 bytes per clock and CU, take the same time (123 us at
// N = 8192 with 768 codebooks and columns, at 2.4 GHz).  Everything else a lane does per codebook adds to the first, so there is little of it:
//   * a slice of the table is [codebook][16-byte piece of the 16 columns][row][16 bytes] (32 rows: 8-byte pieces), 256
//     bytes of a piece being all 64 banks once: no index pattern conflicts, and the piece and the codebook are immediate
//     offsets of the read.  The address is the row number times 16, one bit-field extract from an index word whose nibbles
//     were shifted into place eight at a time;
//   * slices go to LDS with global_load_lds (no registers, no writes), one slice ahead, one barrier per slice;
//   * the reads of several codebooks are in flight while the oldest one's entries are added.
// Measured (us; before: padded rows through registers, two tokens per lane; same bits): N = 8192, 3072 -> 768, 16 centroids
// 223 -> 190 (65 % of the additions' rate), 32 centroids 266 -> 232; N = 12608, 768 -> 3072 343 -> 309; N = 600 3072 -> 768
// 62 -> 27, 32 centroids 89 -> 49; N = 64 60 -> 25.
//
// GROUPED (int8 table with one scale per `group` consecutive codebooks; not in the reference): the table holds the int8
// entries converted to fp32, so the sum inside a group is an exact integer (|sum| <= 128 * group < 2^24 is checked at
// creation); at the end of each group
//     tot = tot + (float)acc_g * scale[g]      (two separately rounded operations, groups ascending)
// and out = tot + bias[f].
#include "gather_common.h"

namespace pimdl {
namespace {

constexpr int F32_THREADS = 256;
typedef int v2i __attribute__((ext_vector_type(2)));

template <int OFF>
__device__ __forceinline__ void lds_read_row(v4i& dst, uint32_t addr)
{
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}
template <int OFF>
__device__ __forceinline__ void lds_read_row(v2i& dst, uint32_t addr)
{
    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}

constexpr int f32_slice_cbs(int c_t) { return c_t == 32 ? 8 : 16; }
constexpr int f32_lds_bytes(int c_t) { return 2 * f32_slice_cbs(c_t) * c_t * 64; }

// A lane is one token with all 16 columns, a workgroup 256 tokens -- or (SPLIT) one token with 4 columns, a workgroup 64
// tokens: the four waves share the columns out, a quarter of the chain of additions, for launches of too few tokens to
// fill the chip the other way.  (Two tokens per lane, a slice serving 512: within 4 % either way at N >= 5000, a chain
// twice as long below.)
template <int C_T, int IDX_BITS, bool GROUPED, bool SPLIT>
__global__ __launch_bounds__(F32_THREADS, 4) void gather_f32_rows_kernel(
    const uint8_t* __restrict__ idx, const float* __restrict__ lut, float* __restrict__ out, uint32_t N, uint32_t M,
    uint32_t CB_pad, uint32_t idx_row_bytes, const float* __restrict__ bias, const float* __restrict__ scales, uint32_t CB,
    uint32_t group, uint32_t act, uint32_t n_token_tiles, uint32_t by_xcd)
{
    constexpr int COLS = SPLIT ? 4 : 16;           // columns of a lane
    constexpr int GS = f32_slice_cbs(C_T), CBB = C_T * 64, SLICE = GS * CBB;
    constexpr int CH = C_T == 32 ? 8 : 16;         // bytes of a read
    constexpr int RD = COLS * 4 / CH;              // reads per codebook
    constexpr int DEPTH = RD == 8 ? 2 : RD == 4 ? 3 : RD == 2 ? 6 : 12;  // codebooks in flight
    constexpr int OPS = SLICE / 1024 / 4;          // copy operations of a wave per slice
    using Row = std::conditional_t<CH == 16, v4i, v2i>;
    static_assert((DEPTH - 1) * RD <= 15 && GS >= DEPTH && OPS >= 1, "the LDS counter; a full pipeline");

    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Workgroup p of the 1-D grid: column block p / n_token_tiles, token tile p % n_token_tiles -- or, by_xcd: workgroups go to the 8
    // XCDs round-robin, and XCD p % 8 takes every token tile of the column blocks congruent to it, so that a column block's part of
    // the table is streamed through one L2 instead of all eight (column blocks past the last: nothing to do).
    const uint32_t pq = by_xcd ? blockIdx.x / 8 : blockIdx.x;
    const uint32_t tile = pq % n_token_tiles;
    const uint32_t colblk = by_xcd ? blockIdx.x % 8 + 8 * (pq / n_token_tiles) : pq / n_token_tiles;
    if (colblk * 16 >= M) return;  // whole workgroup
    const uint32_t tok = SPLIT ? tile * 64 + lane : tile * F32_THREADS + threadIdx.x;
    const uint32_t nslices = CB_pad / GS;  // even
    // 16 bytes of an index row are the codebooks of two slices
    const uint4* idx_row = reinterpret_cast<const uint4*>(idx + (size_t)(tok < N ? tok : N - 1) * idx_row_bytes);

    const uint8_t* src = reinterpret_cast<const uint8_t*>(lut) + (size_t)colblk * CB_pad * CBB + wave * (OPS * 1024) + lane * 16;
    auto copy = [&](uint32_t s, auto bufc) {
        constexpr int buf = decltype(bufc)::value;
        const uint8_t* p = src + (size_t)s * SLICE;
        static_for<0, OPS>([&](auto oc) {
            constexpr int o = decltype(oc)::value;
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)p,
                                             (__attribute__((address_space(3))) void*)(smem + buf * SLICE + wave * (OPS * 1024)), 16, o * 1024, 0);
        });
    };

    float acc[COLS];
    float tot[GROUPED ? COLS : 1];
#pragma unroll
    for (int i = 0; i < COLS; ++i) acc[i] = 0.0f;
#pragma unroll
    for (int i = 0; i < (GROUPED ? COLS : 1); ++i) tot[i] = 0.0f;
    uint32_t cb = 0, in_group = 0, gi = 0;  // workgroup-uniform position in the codebook sequence

    uint4 cur, nxt;
    const uint32_t base = SPLIT ? wave * (RD * C_T * CH) : 0;  // this wave's pieces
    // one slice: two of the four index words in `cur`
    auto slice = [&](auto bufc) __attribute__((always_inline)) {
        constexpr int buf = decltype(bufc)::value;
        // row offsets, ready to be cut out: nibbles * 16 in the bytes of (lo, hi), bytes * 8 in place
        uint32_t lo[2], hi[2];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const uint32_t word = buf == 0 ? (w == 0 ? cur.x : cur.y) : (w == 0 ? cur.z : cur.w);
            if constexpr (IDX_BITS == 4) {
                lo[w] = (word << 4) & 0xF0F0F0F0u;
                hi[w] = word & 0xF0F0F0F0u;
            } else {
                lo[w] = word << 3;  // (ids below 32)
                hi[w] = 0;
            }
        }
        Row ring[DEPTH][RD];
        auto request = [&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;  // codebook of the slice
            constexpr int w = IDX_BITS == 4 ? k / 8 : k / 4, byte = IDX_BITS == 4 ? k % 8 / 2 : k % 4;
            const uint32_t word = (IDX_BITS == 4 && k % 2) ? hi[w] : lo[w];
            // (as assembly, like the pins on the sums below: left free, the compiler makes a slice's addresses up front and
            // its additions at the end, and spills)
            uint32_t addr;
            asm volatile("v_bfe_u32 %0, %1, %2, 8" : "=v"(addr) : "v"(word), "n"(8 * byte));
            if constexpr (SPLIT) addr += base;
            static_for<0, RD>([&](auto rc) {
                constexpr int r = decltype(rc)::value;
                lds_read_row<buf * SLICE + k * CBB + r * C_T * CH>(ring[k % DEPTH][r], addr);
            });
        };
        static_for<0, DEPTH - 1>([&](auto kc) { request(kc); });
        static_for<0, GS>([&](auto kc) {
            constexpr int k = decltype(kc)::value, slot = k % DEPTH;
            if constexpr (k + DEPTH - 1 < GS) request(std::integral_constant<int, k + DEPTH - 1>{});
            constexpr int behind = (GS - 1 - k < DEPTH - 1 ? GS - 1 - k : DEPTH - 1) * RD;  // reads issued after this codebook's
            asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(behind) : "memory");
#pragma unroll
            for (int r = 0; r < RD; ++r) {
                asm volatile("" : "+v"(ring[slot][r]));
#pragma unroll
                for (int e = 0; e < CH / 4; ++e)
                    acc[r * (CH / 4) + e] = __fadd_rn(acc[r * (CH / 4) + e], __int_as_float(ring[slot][r][e]));
            }
#pragma unroll
            for (int i = 0; i < COLS; ++i) asm volatile("" : "+v"(acc[i]));
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (GROUPED) {
                // codebooks past CB are padding (zero rows) and belong to no group
                if (cb < CB && (++in_group == group || cb + 1 == CB)) {
                    const float sc = scalar_load1(scales + gi);
#pragma unroll
                    for (int i = 0; i < COLS; ++i) {
                        tot[i] = __fadd_rn(tot[i], __fmul_rn(acc[i], sc));
                        acc[i] = 0.0f;
                    }
                    ++gi;
                    in_group = 0;
                }
                ++cb;
            }
        });
    };
    // this wave's share of the slice in `buf` has landed; after the barrier everybody's has, and everybody is done with the
    // other buffer
    auto arrive = [&]() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr std::integral_constant<int, 0> b0;
    constexpr std::integral_constant<int, 1> b1;
    copy(0, b0);
    cur = idx_row[0];
    for (uint32_t s = 0; s < nslices; s += 2) {
        arrive();
        nxt = idx_row[s + 2 < nslices ? s / 2 + 1 : s / 2];
        copy(s + 1, b1);
        __builtin_amdgcn_sched_barrier(0);
        slice(b0);
        arrive();
        if (s + 2 < nslices) copy(s + 2, b0);
        __builtin_amdgcn_sched_barrier(0);
        slice(b1);
        cur = nxt;
    }

    if (tok >= N) return;
    const bool vec_store = (M % 4 == 0);  // then every 4-column piece is whole and 16-byte aligned
#pragma unroll
    for (int c = 0; c < COLS / 4; ++c) {
        const uint32_t f = colblk * 16 + (SPLIT ? 4 * wave : 0) + 4 * c;
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            o[e] = activate(__fadd_rn(GROUPED ? tot[4 * c + e] : acc[4 * c + e], (bias && f + e < M) ? bias[f + e] : 0.0f), act);
        if (vec_store) {
            if (f < M) *reinterpret_cast<float4*>(out + (size_t)tok * M + f) = make_float4(o[0], o[1], o[2], o[3]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (f + e < M) out[(size_t)tok * M + f + e] = o[e];
        }
    }
}

// Outputs beyond the last cache in rows of whole 8 KiB: their columns fall on few memory channels, and 256 rows at a time
// (a wave's stores of the whole form, times the column blocks under way) thrash what holds them.  Workgroups of 64 rows, an XCD its own columns,
// write 590 MB in 0.54 ms instead of 1.5 (us, whole in order / whole by XCD / split by XCD: 1 codebook of 16 centroids, M = 4096 N = 36000
// 1502 / 1234 / 541, N = 20000 496 / 597 / 315, M = 2048 N = 36000 320 / 400 / 267; 96 codebooks 8 centroids 1222 / 1338 / 754, 443 /
// 615 / 412, 382 / 393 / 374, 16 centroids 1258 / 1316 / 932, 518 / 627 / 531, 454 / 400 / 490, 32 centroids 1684 / 1332 / 1432, 759 / 699 /
// 868, 672 / 543 / 780; 32 codebooks 32 centroids 1302 / 1321 / 694, 441 / 617 / 394, 356 / 391 / 346; a scale per 8, M = 2048 N = 36000,
// 96 codebooks of 8 centroids 424 / 394 / 583, 64 of 16 379 / 401 / 529).  Below: 12608 x 4096 172 / 266 /
// 182; other widths: 36000 x 3072 364 / 464 / 423, x 4095 680 / 680 / 799.
bool rows_of_8k(const Amm& a, uint32_t n)
{
    const uint64_t out_bytes = (uint64_t)n * a.g.M * 4;
    return a.g.M % 2048 == 0 && out_bytes > (256ull << 20) && a.lut_bytes < out_bytes;
}

template <int C_T, int IDX_BITS, bool GROUPED, bool SPLIT>
int launch_f32_as(Ctx* ctx, const Amm& a, const uint8_t* d_idx, float* d_out, uint32_t n)
{
    constexpr int LDS = f32_lds_bytes(C_T);
    constexpr uint32_t TOKENS = SPLIT ? 64 : F32_THREADS;
    auto kern = gather_f32_rows_kernel<C_T, IDX_BITS, GROUPED, SPLIT>;
    if (int rc = allow_dynamic_lds(ctx, reinterpret_cast<const void*>(kern), LDS, "hipFuncSetAttribute(gather_f32)")) return rc;
    const uint32_t n_token_tiles = (n + TOKENS - 1) / TOKENS, colblocks = a.g.M_pad / 16;
    // By XCD where the table's traffic counts and the column blocks divide evenly enough (an eighth more at most).  Not for outputs
    // beyond the caches, and larger than the table, in rows of more than 4 KiB of whole float4s: eight column blocks side by side then
    // write pieces of the same rows at the same time (us, by XCD / in order: 16 centroids, 1 codebook, N = 27003, M = 3072 358 / 252;
    // 64 codebooks, N = 6664, M = 4096 127 / 102; 192 codebooks, N = 12608, M = 3072 291 / 292, N = 2048 61 / 64; 32 centroids, 256
    // codebooks, N = 2048, M = 3072 86 / 116, N = 6664, M = 4096 347 / 375; 768 codebooks, N = 12608, M = 768 368 / 488; odd widths,
    // 128 codebooks, N = 9919, M = 4095 317 / 344; rows of up to 4 KiB, 1 codebook, 180 MB, M = 512 130 / 177, M = 1024 147 / 196,
    // M = 768 135 / 134; few tokens, 192 codebooks, N = 328, M = 2157 26 / 53).
    // Rows of whole 8 KiB that together exceed the last cache are the exception: by XCD, in the split form where its chain is short and
    // with 32 centroids (rows_of_8k).  Uneven column blocks of the whole form only where the CUs of an XCD take at most an eighth more
    // rounds (8 centroids, a scale per 8 of 96 codebooks, N = 6444, M = 608, 38 column blocks 41.5 / 34.4).
    const uint64_t out_bytes = (uint64_t)n * a.g.M * 4;
    const uint64_t padded = (colblocks + 7) / 8 * 8, cus = ctx->prop.multiProcessorCount;
    const bool wide_output = a.g.M % 4 == 0 && a.g.M > 1024 && out_bytes >= (40ull << 20) && a.lut_bytes < out_bytes &&
                             !((SPLIT || C_T == 32) && rows_of_8k(a, n));
    const bool even = 8 * (padded - colblocks) <= colblocks &&
                      (SPLIT || 8 * ((n_token_tiles * padded + cus - 1) / cus) <= 9 * (((uint64_t)n_token_tiles * colblocks + cus - 1) / cus));
    const uint32_t by_xcd = even && !wide_output ? 1u : 0u;
    const uint64_t wgs = (uint64_t)n_token_tiles * (by_xcd ? padded : colblocks);
    if (wgs > 0x7FFFFFFFull) return set_error(ctx, PIMDL_ERR_UNSUPPORTED, "gather: %llu workgroups", (unsigned long long)wgs);
    snprintf(a.last_gather, sizeof(a.last_gather), "gather_f32_rows_kernel<%d, %d, %s, %s>", C_T, IDX_BITS, GROUPED ? "true" : "false",
             SPLIT ? "true" : "false");
    a.note_launch(f32_slice_cbs(C_T), LDS, TOKENS, F32_THREADS);
    hipLaunchKernelGGL(kern, dim3((uint32_t)wgs), dim3(F32_THREADS), LDS, ctx->stream, d_idx, reinterpret_cast<const float*>(a.d_lut),
                       d_out, n, a.g.M, a.g.CB_pad, a.g.idx_row_bytes, a.d_bias, a.d_scales, a.g.CB, a.desc.scale_group,
                       a.desc.activation, n_token_tiles, by_xcd);
    return hip_check(ctx, hipGetLastError(), "gather_f32_rows_kernel launch");
}

// Which of the two is the shorter launch: w, w1 workgroups per CU of either form.  The split form's chain takes 0.57 of the
// other's and its time grows from two workgroups per CU on (four with the half-size slices of 8 rows), the other's from
// one.  us, split / whole: 768 -> 3072, 16 centroids N = 64 8.9 / 13.4, 300 15.8 / 19.7, 600 28.8 / 28.0, 1200 53 / 40; 3072 ->
// 768 N = 64 25 / 42, 600 27 / 44, 1200 52 / 46, 8192 273 / 190; 8 centroids, 1024 -> 1024 N = 600 12 / 18, 1200 20 / 23,
// 2500 38 / 37; 32 centroids (whose slices take longer to copy than to add, which two workgroups of the whole form share),
// 768 -> 768 N = 600 12 / 19, 1200 23 / 21; 192 codebooks, M = 2048 N = 283 18.5 / 18.4, M = 4096 N = 130 19.5 / 19.8, 283 33 / 23;
// 768 codebooks, M = 3370 N = 283 158 / 87.  A scale per group is work per codebook whatever the columns: 8 centroids, a
// scale per 8, 192 codebooks, M = 3072 N = 300 31 / 34, 600 46 / 38, 1200 71 / 49, 768 codebooks, M = 768 N = 1200 94 / 102, 2500 152 / 104, 3080
// 180 / 119.
template <int C_T, int IDX_BITS, bool GROUPED>
int launch_f32(Ctx* ctx, const Amm& a, const uint8_t* d_idx, float* d_out, uint32_t n)
{
    const double per_cu = (double)(a.g.M_pad / 16) / ctx->prop.multiProcessorCount;
    const double w = (n + 63) / 64 * per_cu, w1 = (n + F32_THREADS - 1) / F32_THREADS * per_cu;
    const double grow = (C_T == 8 ? (GROUPED ? 0.49 : 0.42) : 0.58) * w, grow1 = C_T == 32 ? 0.5 * w1 + 0.4 : 0.85 * w1 + 0.15;
    const bool short_chain = a.g.CB_pad <= (C_T == 32 ? 32u : C_T == 8 ? (GROUPED ? 64u : 96u) : (GROUPED ? 32u : 64u));
    if ((short_chain && rows_of_8k(a, n)) || 0.57 * (grow > 1 ? grow : 1) < (grow1 > 1 ? grow1 : 1))
        return launch_f32_as<C_T, IDX_BITS, GROUPED, true>(ctx, a, d_idx, d_out, n);
    return launch_f32_as<C_T, IDX_BITS, GROUPED, false>(ctx, a, d_idx, d_out, n);
}

}  // namespace

uint32_t f32_rows_lds_bytes(uint32_t c_tile) { return (uint32_t)f32_lds_bytes((int)c_tile); }

int launch_gather_f32_rows(Ctx* ctx, const Amm& a, const uint8_t* d_idx, float* d_out, uint32_t n)
{
    const bool bounds = a.grouped && !a.prescaled;  // a scale to apply at the end of every group
    switch (a.g.C_tile) {
        case 8: return bounds ? launch_f32<8, 4, true>(ctx, a, d_idx, d_out, n) : launch_f32<8, 4, false>(ctx, a, d_idx, d_out, n);
        case 16: return bounds ? launch_f32<16, 4, true>(ctx, a, d_idx, d_out, n) : launch_f32<16, 4, false>(ctx, a, d_idx, d_out, n);
        case 32: return bounds ? launch_f32<32, 8, true>(ctx, a, d_idx, d_out, n) : launch_f32<32, 8, false>(ctx, a, d_idx, d_out, n);
    }
    return set_error(ctx, PIMDL_ERR_UNSUPPORTED, "no fp32 row gather for C_tile=%u", a.g.C_tile);
}

}  // namespace pimdl
