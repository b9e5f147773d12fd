// LUT gather-accumulate by reading rows from LDS (gfx950), int8 tables: the kernel for 17 centroids and more.
//
// Same operator as the other gather kernels (inference-engine/src/dpu/pim_lut_kernel.c:97-2296, row-major
// statement inference-engine/test/test_amm.cpp:164-175, epilogue inference-engine/src/host/pim_lut_host.cpp:190-203):
//     acc[n][f] = sum over cb of lut[cb][idx[n][cb]][f]          (int8 table, int32 sum, exact)
// Every gathered byte is read from LDS once, N * CB * M bytes whatever the number of centroids, and the matrix
// core adds the bytes: v_smfmac_i32_16x16x128_i8 with a constant sparse operand A[i][16 k + b] = (b == i) -- one
// non-zero in sixteen, a valid 2:4 pattern -- and the gathered row pieces as the dense operand computes
//     D[i][j] += sum over k = 0..7 of byte i of token j's k-th row piece,
// i.e. ONE instruction adds 2048 gathered bytes into int32 accumulators (twice what the dense
// v_mfma_i32_16x16x64_i8 does at the same issue rate).  No work is multiplied by the number of centroids.
//
// What bounds it is the LDS: 256 bytes per clock and CU, if no two lanes that are served together meet in a bank.
// A ds_read_b128 is served in four passes of 16 lanes over 64 banks, so the 16 lanes of a pass have to read 16
// different 16-byte columns of banks, and their rows are whatever the tokens' indices are.  So a pass reads 16
// DIFFERENT codebooks, and every codebook owns a column of banks: the table slice of 16 codebooks and 16 output
// columns is laid out [row][codebook][16 bytes] (a row of 256 bytes is all 64 banks once), and token j reads
// codebook j ^ x at step x = 0..15.  Over the steps every token meets every codebook of the slice (the order of an
// integer sum is free), and in each step the 16 tokens of a pass stand in 16 different bank columns, whatever the
// indices.  (Rows of one codebook side by side, as before, are free of conflicts up to 16 rows only: 64 centroids
// met two to three deep in a bank, 140 us at N = 8192, 768 -> 3072 where the reads alone are 31 us.)
//
// The passes are lanes {0-3,12-15,20-27}, {4-11,16-19,28-31}, {32-35,44-47,52-59}, {36-43,48-51,60-63} (measured):
// each holds all 16 tokens j = lane % 16, taken from two of the four lane groups lane / 16.  A lane's steps are
// x = 4 * pass + 0..3, so its four codebooks j ^ x are the four of ONE quarter of the slice, (j >> 2) ^ pass, in an
// order that depends on j: with one-byte indices they are one 32-bit word of the packed index row.
//
// Measured (us; before: rows of one codebook side by side, dense matrix instruction; the floor is N * CB * M bytes at
// 256 bytes per clock, CU and 2.4 GHz): N = 8192, 768 -> 3072, v = 4: 64 centroids 140 -> 61, 128 186 -> 74, 256
// 338 -> 83 (floor 31); N = 12608, 32 centroids (before: the sparse one-hot kernel) 768 -> 3072 119 -> 94, 3072 -> 768
// 122 -> 93 (floor 47).  Counters: no bank conflicts, LDS busy 63 % of the CUs' cycles at 64
// centroids and 73 % at 32; the rest is the copies of the slices (43 bytes per clock and CU), the barriers and the last items of
// the grid.
//
// Table in HBM: [16-column chunk][slice of 16 codebooks][row][codebook][16 columns], so a slice of a chunk is one
// contiguous block that goes to LDS with global_load_lds (no registers).  An item is NW * TG * 16 tokens x Q chunks.
#include "gather_common.h"

namespace pimdl {
namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
// four columns of a row of any width: 16-byte stores need dword alignment only
typedef float v4f_dw __attribute__((ext_vector_type(4), aligned(4)));
typedef int v4i_dw __attribute__((ext_vector_type(4), aligned(4)));

template <int N>
__device__ __forceinline__ void lgkm_wait()
{
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N < 15 ? N : 15) : "memory");
}

constexpr int rw_lds_bytes(int c_t, int q) { return 2 * q * c_t * 256; }  // two slice buffers
constexpr int rw_wgs_per_cu(int nw) { return nw == 8 ? 2 : 1; }           // four waves per SIMD either way

// C_T: rows of a codebook in the table (>= centroids); Q: 16-column chunks per item; NW: waves; TG: 16-token groups
// per wave; WPS: waves per SIMD the registers are cut for
template <int C_T, int Q, int NW, int TG, int WPS, int IDX_BITS>
__global__ __launch_bounds__(NW * 64, WPS) void gather_i8_kernel(
    const uint8_t* __restrict__ idx, const int8_t* __restrict__ lut, float* __restrict__ out,
    int32_t* __restrict__ acc_out, uint32_t N, uint32_t M, uint32_t nslices, uint32_t table_slices, uint32_t nchunks, uint32_t idx_row_bytes,
    uint32_t n_token_tiles, uint32_t n_items, Epilogue ep, XcdMap xmap)
{
    constexpr int CHUNK = C_T * 256;               // bytes of one slice of one chunk
    constexpr int SLICE = Q * CHUNK;
    constexpr int TOK_ITEM = NW * TG * 16;
    constexpr int NBLK = SLICE / 1024;             // 1 KB blocks (one copy instruction of a wave) per slice
    constexpr int BPC = CHUNK / 1024;              // ... per chunk
    constexpr int BPW = (NBLK + NW - 1) / NW;      // ... per wave
    static_assert((Q - 1) * CHUNK < 65536, "chunk offsets fit the immediate of ds_read");

    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t j = lane & 15;  // token within a 16-token group
    const uint32_t g = lane >> 4;  // which 4 of a chunk's 16 columns this lane ends up with
    const uint32_t pass = g ^ (((j + 4) >> 3) & 1);
    if (blockIdx.x >= n_items) return;  // whole workgroup
    const uint32_t my_items = (n_items - blockIdx.x + gridDim.x - 1) / gridDim.x;
    const uint32_t total = my_items * nslices;

    // constant sparse operand: per block of 16 positions, value 1 at position j -- first value slot of group j / 4,
    // position j % 4 (both blocks of the lane alike)
    const uint64_t one = 1ull << (16 * (j >> 2));
    const v4i a_sel = {(int)(uint32_t)one, (int)(uint32_t)(one >> 32), (int)(uint32_t)one, (int)(uint32_t)(one >> 32)};
    const int a_pos = (int)(((j & 3) << (4 * (j >> 2))) * 0x10001u);

    // step s = 0..3 reads codebook q = j ^ (4 pass + s) of the slice: its 16-byte column of banks starts at 16 q of a
    // row, and its index sits IDX_BITS * (q % (32 / IDX_BITS)) bits into the lane's index word; both follow from
    // step 0's by flipping the bits of s
    const uint32_t q0 = j ^ (4 * pass);
    const uint32_t shift0 = IDX_BITS * (q0 & (32 / IDX_BITS - 1));
    const uint32_t idx_word = IDX_BITS == 8 ? (j >> 2) ^ pass : (j >> 3) ^ (pass >> 1);
    // the index words of a token block's tail, past the last token, are not written by anyone: masked to the table's rows
    constexpr int ROW_BITS = C_T == 16 ? 4 : C_T == 32 ? 5 : C_T == 64 ? 6 : C_T == 128 ? 7 : 8;
    static_assert(C_T == 1 << ROW_BITS, "rows of a codebook");
    constexpr uint32_t SLICE_WORDS = 16 * IDX_BITS / 32;  // index words per token and slice

    auto col_of = [&](uint32_t p) { uint32_t c, t; xmap.decode(p, n_token_tiles, c, t); return c; };
    auto tok_tile_of = [&](uint32_t p) { uint32_t c, t; xmap.decode(p, n_token_tiles, c, t); return t; };

    // ---- streams: the slice being copied (one ahead of the one being read) and its index words --------------
    uint32_t nx_item = blockIdx.x, nx_s = 0;
    const int8_t* cp_base;           // uniform: slice 0 of the first chunk of the copied item
    uint32_t cp_chunk0;              // its first chunk
    constexpr int TB = TG > 4 ? TG / 4 : 1;  // 64-token index blocks of a wave
    const uint8_t* ix_base[TB];      // uniform: the wave's tokens in the index words of slice 0 of the copied item
    const uint32_t ix_lane = idx_word * 256 + j * 4;
    const size_t chunk_stride = (size_t)table_slices * CHUNK;
    const uint32_t last_block = (N - 1) / 64;
    auto locate = [&]() __attribute__((always_inline)) {
        uint32_t col, tile;
        xmap.decode(nx_item, n_token_tiles, col, tile);
        cp_chunk0 = col * Q;
        cp_base = lut + (size_t)cp_chunk0 * chunk_stride;
        const uint32_t op = ep.op_col_tiles ? col / ep.op_col_tiles : 0u;
        const uint32_t tok0 = tile * TOK_ITEM + wave * (TG * 16);
#pragma unroll
        for (int b = 0; b < TB; ++b) {
            uint32_t blk = tok0 / 64 + b;
            if (blk > last_block) blk = last_block;  // clamp: results of such tokens are never stored
            ix_base[b] = idx + (size_t)op * ep.op_idx_stride + (size_t)blk * idx_row_bytes * 64 + (tok0 & 63) * 4;
        }
    };
    auto stage = [&](uint32_t buf_off) __attribute__((always_inline)) {  // slice nx_s of item nx_item into a buffer
#pragma unroll
        for (int u = 0; u < BPW; ++u) {
            const uint32_t b = wave * BPW + u;
            if (NBLK % NW != 0 && b >= NBLK) continue;  // wave-uniform
            uint32_t c = b / BPC;
            const uint32_t dst = buf_off + b * 1024;
            if (cp_chunk0 + c >= nchunks) c = nchunks - 1 - cp_chunk0;  // past the last chunk: never stored
            const int8_t* src = cp_base + (size_t)c * chunk_stride + (size_t)nx_s * CHUNK + (b % BPC) * 1024;
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + lane * 16),
                                             (__attribute__((address_space(3))) void*)(smem + dst), 16, 0, 0);
        }
    };
    auto advance = [&]() __attribute__((always_inline)) {
        if (++nx_s == nslices) {
            nx_s = 0;
            nx_item += gridDim.x;
            if (nx_item < n_items) locate();
        }
    };

    v4i acc[TG][Q];
#pragma unroll
    for (int t = 0; t < TG; ++t)
#pragma unroll
        for (int c = 0; c < Q; ++c) acc[t][c] = (v4i){0, 0, 0, 0};

    // ---- epilogue: lane (j, g) holds columns 4 g .. 4 g + 3 of every chunk for token j of every group --------
    // All bias values first, then the stores row by row: with a chunk's bias loaded behind the chunk before it, every chunk waited for
    // the stores so far, and the rows were written in Q passes (us, before / now: one codebook, N = 38004, M = 3131, 16 centroids
    // 354 / 249, 64 centroids 338 / 275; N = 25265, M = 3072, 96 codebooks, 64 centroids 160 / 139).  Four columns in one store at any
    // width (us, float by float where M % 4 != 0 / now: 32 centroids, N = 20000, M = 1001, 1 codebook 49 / 27, 192 codebooks 76 / 56;
    // 64 centroids, N = 38004, M = 3131, 33 codebooks 349 / 281).
    auto epilogue_as = [&](uint32_t item, auto actc) __attribute__((always_inline)) {
        constexpr bool ACT = decltype(actc)::value;
        const uint32_t col = col_of(item);
        Epilogue epl = ep;
        if (ep.op_col_tiles) epl.scale = scalar_load1(ep.op_scales + col / ep.op_col_tiles);
        // (opaque, so that none of the address arithmetic is kept in registers through the slices)
        uint32_t je = j, ge = g;
        asm volatile("" : "+v"(je), "+v"(ge));
        const uint32_t tok0 = tok_tile_of(item) * TOK_ITEM + wave * (TG * 16) + je;
        float bv[Q][4];
#pragma unroll
        for (int c = 0; c < Q; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t f = (col * Q + c) * 16 + 4 * ge + e;
                bv[c][e] = (ep.bias && f < M) ? ep.bias[f] : 0.0f;
            }
#pragma unroll
        for (int t = 0; t < TG; ++t) {
            const uint32_t tok = tok0 + t * 16;
#pragma unroll
            for (int c = 0; c < Q; ++c) {
                const uint32_t f = (col * Q + c) * 16 + 4 * ge;
                const v4i a = acc[t][c];
                acc[t][c] = (v4i){0, 0, 0, 0};
                if (tok >= N || f >= M) continue;
                float o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = dequant<ACT>(a[e], epl, bv[c][e]);
                const size_t at = (size_t)tok * M + f;
                if (f + 4 <= M) {
                    *reinterpret_cast<v4f_dw*>(out + at) = (v4f_dw){o[0], o[1], o[2], o[3]};
                    if (acc_out) *reinterpret_cast<v4i_dw*>(acc_out + at) = (v4i_dw){a[0], a[1], a[2], a[3]};
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (f + e < M) {
                            out[at + e] = o[e];
                            if (acc_out) acc_out[at + e] = a[e];
                        }
                }
            }
        }
    };
    auto epilogue = [&](uint32_t item) __attribute__((always_inline)) {
        if (ep.act == PIMDL_ACT_GELU_TANH) epilogue_as(item, std::true_type{});
        else epilogue_as(item, std::false_type{});
    };

    // ---- prologue: slice 0 ------------------------------------------------------------------------------------
    locate();
    uint32_t word[TG], word_nxt[TG];
    auto load_words = [&]() __attribute__((always_inline)) {
        const size_t at = (size_t)nx_s * SLICE_WORDS * 256;
#pragma unroll
        for (int t = 0; t < TG; ++t)
            word_nxt[t] = *reinterpret_cast<const uint32_t*>(ix_base[t / 4] + at + ix_lane + t % 4 * 64);
    };
    stage(0);
    load_words();
    advance();

    uint32_t k = 0, buf = 0;
    for (uint32_t item0 = blockIdx.x; item0 < n_items; item0 += gridDim.x) {
        for (uint32_t s0 = 0; s0 < nslices; ++s0, ++k) {
            // this wave's copies of slice k and its index words have landed; after the barrier everybody's have, and
            // everybody is done with slice k - 1, whose buffer slice k + 1 goes into
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
            for (int t = 0; t < TG; ++t) word[t] = word_nxt[t];
            __syncthreads();
            if (k + 1 < total) {
                stage(buf ^ SLICE);
                load_words();
                advance();
            }
            __builtin_amdgcn_sched_barrier(0);

            // Pair p = (token group, half of the lane's four steps, chunk): two reads, one matrix instruction.  D
            // pairs are in flight; LDS operations complete in order, so the wait counts what was issued behind.
            constexpr int P = TG * 2 * Q, D = P < 3 ? P : 3;
            v4i lo[D], hi[D];
            uint32_t addr[2];
            const uint32_t base0 = 16 * q0 + buf;
            auto issue = [&](auto pc) __attribute__((always_inline)) {
                constexpr int p = decltype(pc)::value, c = p % Q, h = p / Q % 2, t = p / Q / 2;
                if constexpr (c == 0) {
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const uint32_t x = 2 * h + e;
                        addr[e] = (__builtin_amdgcn_ubfe(word[t], shift0 ^ (IDX_BITS * x), ROW_BITS) << 8) + (base0 ^ (16 * x));
                    }
                }
                lds_read<c * CHUNK>(lo[p % D], addr[0]);
                lds_read<c * CHUNK>(hi[p % D], addr[1]);
            };
            static_for<0, D>([&](auto pc) { issue(pc); });
            static_for<0, P>([&](auto pc) {
                constexpr int p = decltype(pc)::value, c = p % Q, t = p / Q / 2;
                constexpr int behind = P - 1 - p < D - 1 ? P - 1 - p : D - 1;
                lgkm_wait<2 * behind>();
                asm volatile("" : "+v"(lo[p % D]), "+v"(hi[p % D]));
                __builtin_amdgcn_sched_barrier(0);
                const v4i l = lo[p % D], h4 = hi[p % D];
                const v8i bb = {l[0], l[1], l[2], l[3], h4[0], h4[1], h4[2], h4[3]};
                acc[t][c] = __builtin_amdgcn_smfmac_i32_16x16x128_i8(a_sel, bb, acc[t][c], a_pos, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (p + D < P) issue(std::integral_constant<int, p + D>{});
            });
            buf ^= SLICE;
        }
        epilogue(item0);
    }
}

struct RowsLaunch {
    Ctx* ctx;
    const Amm& a;
    const uint8_t* d_idx;
    float* d_out;
    int32_t* d_acc;
    uint32_t n;
    Epilogue ep;
};

// Shape of an item: NW * TG * 16 tokens x Q chunks, two workgroups of eight waves per CU or one of sixteen.
template <int Q_, int NW_, int TG_>
struct RowsShape {
    static constexpr int Q = Q_, NW = NW_, TG = TG_, TOKENS = NW_ * TG_ * 16;
};

template <int C_T, int IDX_BITS, class S>
int launch_rows_as(const RowsLaunch& l)
{
    constexpr int LDS = rw_lds_bytes(C_T, S::Q), WPS = 4;
    static_assert(rw_wgs_per_cu(S::NW) * LDS <= 160 * 1024, "the CU's LDS holds the workgroups that its registers hold");
    const AmmGeom& g = l.a.g;
    auto kern = gather_i8_kernel<C_T, S::Q, S::NW, S::TG, WPS, IDX_BITS>;
    if (int rc = allow_dynamic_lds(l.ctx, reinterpret_cast<const void*>(kern), LDS, "hipFuncSetAttribute(gather_i8)")) return rc;
    const uint32_t n_token_tiles = (l.n + S::TOKENS - 1) / S::TOKENS;
    const uint32_t nchunks = g.M_pad / 16, col_tiles = (nchunks + S::Q - 1) / S::Q;
    const uint32_t n_items = n_token_tiles * col_tiles;
    uint32_t grid = l.ctx->prop.multiProcessorCount * rw_wgs_per_cu(S::NW);
    if (grid > n_items) grid = n_items;
    // Outputs well beyond the last cache, of tables that are small beside them: an XCD writes whole rows (its own token tiles) instead of
    // its own columns of all rows, which would have several XCDs write pieces of the same rows at the same time (us, by the table's
    // traffic / by rows: 24 centroids, N = 36621, M = 3072, 1 codebook 154 / 134, 32 160 / 139, 96 208 / 200; N = 27465, M = 4096, 1
    // codebook 161 / 148; 64 centroids 156 / 135, 157 / 146, 96 codebooks 270 / 261.  Not: 64 centroids, 192 codebooks, N = 36621, M = 2048
    // 281 / 293; tiles of one chunk, 128 centroids, 32 codebooks 240 / 253; outputs of 300 MB, N = 24414, M = 3072 78 / 78).
    const uint64_t table = (uint64_t)g.CB_pad * C_T * g.M_pad, out_bytes = (uint64_t)l.n * g.M * 4;
    const bool by_tokens = S::Q > 1 && out_bytes > (320ull << 20) && table * 16 < out_bytes;
    const uint32_t split = g.tune_xcd_col_split || !by_tokens ? g.tune_xcd_col_split : n_token_tiles % 8 == 0 ? 1u : PIMDL_XCD_PLAIN;
    const XcdMap xmap = choose_xcd_map(col_tiles, n_token_tiles, grid, table, (uint64_t)l.n * g.idx_row_bytes, split);
    Epilogue ep = l.ep;
    ep.op_col_tiles = ep.op_col_tiles * g.q / S::Q;
    snprintf(l.a.last_gather, sizeof(l.a.last_gather), "gather_i8_kernel<%d, %d, %d, %d, %d, %d>", C_T, S::Q, S::NW, S::TG, WPS, IDX_BITS);
    l.a.note_launch(16, LDS, S::TOKENS, S::NW * 64);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(S::NW * 64), LDS, l.ctx->stream, l.d_idx, reinterpret_cast<const int8_t*>(l.a.d_lut),
                       l.d_out, l.d_acc, l.n, g.M, (g.CB + 15) / 16, g.CB_pad / 16, nchunks, g.idx_row_bytes, n_token_tiles, n_items,
                       ep, xmap);
    return hip_check(l.ctx, hipGetLastError(), "gather_i8_kernel launch");
}

// Clocks of a launch, up to a common factor.  A slice costs its copies (C_T rows x 256 bytes per chunk at about 43
// bytes per clock and CU, measured) and its reads (4 per token group and chunk, 4.08 clocks each, half as much again
// for what the waves do not overlap), and the persistent grid pays for rounds of items (grid_rounds).  Measured
// against this for N = 8192, 768 -> 3072 at 64 centroids (us): 2 chunks x 1024 tokens 60, x 512 70, x 256 85,
// x 128 133; 1 chunk x 1024 69, x 512 80; N = 1024: 2 x 512 16.6, 2 x 256 16.3, 2 x 128 21.6, 1 x 512 15.5.
template <int C_T, class S>
double rows_cost(const RowsLaunch& l)
{
    const AmmGeom& g = l.a.g;
    const uint32_t nchunks = g.M_pad / 16;
    // operators side by side: a tile of columns belongs to one of them
    if (l.ep.op_col_tiles && l.ep.op_col_tiles * g.q % S::Q != 0) return 1e300;
    const uint64_t items = (uint64_t)((l.n + S::TOKENS - 1) / S::TOKENS) * ((nchunks + S::Q - 1) / S::Q);
    const double wgs = rw_wgs_per_cu(S::NW);
    const double slice = wgs * S::Q * (C_T * 256 / 43.0 + S::NW * S::TG * 24.5) + 150;
    return grid_rounds(items, (uint64_t)(wgs * l.ctx->prop.multiProcessorCount)) * ((g.CB + 15) / 16 * slice + 2000);
}

template <int C_T, int IDX_BITS, class... S>
int launch_rows(const RowsLaunch& l)
{
    const double cost[] = {rows_cost<C_T, S>(l)...};
    int (*const launch[])(const RowsLaunch&) = {launch_rows_as<C_T, IDX_BITS, S>...};
    int best = 0;
    for (int i = 1; i < (int)sizeof...(S); ++i)
        if (cost[i] < cost[best]) best = i;
    return launch[best](l);
}

}  // namespace

int launch_gather_rows(Ctx* ctx, const Amm& a, const uint8_t* d_idx, float* d_out, int32_t* d_acc, uint32_t n, float scale,
                       float lut_bias_term)
{
    Epilogue ep;
    ep.scale = scale;
    ep.lut_bias_term = lut_bias_term;
    ep.bias = a.d_bias;
    ep.act = a.desc.activation;
    ep.op_scales = a.d_op_scales;
    ep.op_col_tiles = a.op_col_tiles;
    ep.op_idx_stride = a.op_idx_stride;
    const RowsLaunch l{ctx, a, d_idx, d_out, d_acc, n, ep};
    // A width that the caller has named, and 48 columns for operators side by side that tiles of two and four chunks do not
    // divide; the launch's own choice below.
    if (a.g.cols == 48 || (ep.op_col_tiles * a.g.q) % 2 != 0) {
        switch (a.g.C_tile) {
            case 16: return launch_rows<16, 4, RowsShape<3, 8, 4>, RowsShape<3, 8, 2>, RowsShape<3, 8, 1>>(l);
            case 32: return launch_rows<32, 8, RowsShape<3, 8, 4>, RowsShape<3, 8, 2>, RowsShape<3, 8, 1>>(l);
            case 64: return launch_rows<64, 8, RowsShape<3, 16, 4>, RowsShape<3, 16, 2>, RowsShape<3, 16, 1>>(l);
        }
    } else if (a.g.cols == 64 && a.g.C_tile >= 32) {
        switch (a.g.C_tile) {
            case 32: return launch_rows<32, 8, RowsShape<4, 8, 4>, RowsShape<4, 8, 2>, RowsShape<4, 8, 1>>(l);
            case 64: return launch_rows<64, 8, RowsShape<4, 16, 4>, RowsShape<4, 16, 2>, RowsShape<4, 16, 1>>(l);
        }
    } else {
        switch (a.g.C_tile) {
            case 16: return launch_rows<16, 4, RowsShape<4, 8, 4>, RowsShape<4, 8, 2>, RowsShape<4, 8, 1>>(l);
            case 32:
                return launch_rows<32, 8, RowsShape<2, 8, 8>, RowsShape<4, 8, 4>, RowsShape<2, 8, 4>, RowsShape<2, 8, 2>,
                                   RowsShape<2, 8, 1>>(l);
            case 64:
                return launch_rows<64, 8, RowsShape<2, 8, 8>, RowsShape<2, 8, 4>, RowsShape<1, 8, 4>, RowsShape<1, 8, 2>,
                                   RowsShape<1, 8, 1>>(l);
            case 128:
                return launch_rows<128, 8, RowsShape<1, 8, 8>, RowsShape<2, 16, 4>, RowsShape<1, 8, 4>, RowsShape<1, 8, 2>,
                                   RowsShape<1, 8, 1>>(l);
            case 256:
                return launch_rows<256, 8, RowsShape<1, 16, 8>, RowsShape<1, 16, 4>, RowsShape<1, 16, 2>, RowsShape<1, 16, 1>>(l);
        }
    }
    return set_error(ctx, PIMDL_ERR_UNSUPPORTED, "no row gather kernel for %u centroids x %u chunks", a.g.C_tile, a.g.q);
}

uint32_t rows_lds_bytes(uint32_t c_tile, uint32_t q) { return (uint32_t)rw_lds_bytes((int)c_tile, (int)q); }

}  // namespace pimdl
