// LUT gather-accumulate for launches of few tokens (gfx950): the codebooks are what is dealt out.
//
// Same operator as the other gather kernels (inference-engine/src/dpu/pim_lut_kernel.c:97-2296, row-major
// statement inference-engine/test/test_amm.cpp:164-175, epilogue inference-engine/src/host/pim_lut_host.cpp:190-203):
//     acc[n][f] = sum over cb of lut[cb][idx[n][cb]][f]
// on the tables of the large kernels, whatever their layout.  Those kernels give an item of 128 tokens or more and 16 to
// 96 columns to a workgroup, which goes through all codebooks slice by slice; a launch with fewer items than CUs
// then takes the time of that chain -- copy, barrier, operands, 32 codebooks further -- however few its tokens are.
#include <math.h>
#include <string.h>

#include <algorithm>

#include "gather_common.h"
#include "search_quad.h"

namespace pimdl {
namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v2i __attribute__((ext_vector_type(2)));

// An int8 launch: a workgroup takes 16 columns (32 or 48 of the sparse table between few and many tokens) of 16 * TM tokens, its NW waves deal out the K-steps of the matrix
// instruction, every operand comes straight from memory (nothing is shared between waves, so nothing is staged), and the
// waves' int32 sums meet in LDS once, at the end.  All loads of a wave are in flight together: a launch is one
// round trip for the indices and the table, not one per slice.  What bounds it: up to 16 tokens the launch itself and
// that round trip (3.0 us at 768 -> 3072, 4.5 at 3072 -> 768, whose 9.4 MB of table 48 CUs read; before 8.1 / 19.8);
// beyond, the table entries that every 64 tokens read again and the operands made from index bytes (7.5 us at N = 64).
constexpr int FEW_UNROLL = 4;       // K-steps of a wave whose loads are in flight together
// floats between a wave's registers in the exchange: the reads below meet in no bank
constexpr int FEW_PITCH_ONEHOT = 80, FEW_PITCH_ROWS = 68;
constexpr int few_lds_bytes(int nw, int tm, int pitch) { return nw * tm * 4 * pitch * 4; }

enum FewTable { FEW_SPARSE, FEW_PAIRED, FEW_ROWS };

// What a launch leaves as Amm::last_gather, put together once: these launches are short enough for the host to feel a snprintf.
struct KernelName {
    char text[sizeof(Amm::last_gather)];
    template <class... A>
    explicit KernelName(const char* format, A... args) { snprintf(text, sizeof(text), format, args...); }
    void to(char* last_gather) const { memcpy(last_gather, text, sizeof(text)); }
};

struct FewArgs {
    const uint8_t* idx;
    const int8_t* lut;
    float* out;
    int32_t* acc_out;
    uint32_t N, M;
    uint32_t groups;        // 16-column groups of the table
    uint32_t steps;         // K-steps
    uint32_t tile_groups;   // one-hot tables: 16-column groups per column tile; rows: 1
    uint32_t c_tile;        // rows: rows per codebook in the table
    uint32_t idx_row_bytes;
    uint32_t op_groups;     // operators side by side: 16-column groups of each (0: one operator)
};
// the search of a launch that has no index buffer
struct FewSearch {
    const float* x;
    const float* cent;
    uint32_t K, CB, C, aligned;
};
constexpr int FEW_FUSED_TOKENS = 2;

// Column of position s of a tile of one-hot tables (sparse_tile_column on the device)
__device__ __forceinline__ uint32_t few_column(uint32_t tn, uint32_t c, uint32_t j)
{
    const uint32_t n4 = tn / 4 * 4, n2 = n4 + (tn % 4) / 2 * 2;
    if (c < n4) return 16 * (c / 4 * 4) + 4 * j + c % 4;
    if (c < n2) return 16 * n4 + 2 * j + (c - n4);
    return 16 * c + j;
}

// One workgroup per (16 * TC columns, 16 * TM tokens).  Operands of a K-step, lane l = 16 g + j:
//   FEW_SPARSE  the sparse one-hot product (8 codebooks of 16): lane (g, token j) turns byte g of index word s into value
//               bytes and positions, lane (g, column j) reads the table entries of codebooks g and g + 4
//   FEW_PAIRED  the same instruction on the paired table (up to 8 centroids): an entry's 16 slots are two codebooks of
//               8, whose one-hots fall into different groups of four, so a K-step covers 16 codebooks
//   FEW_ROWS    the byte adder: lane (g, token j) reads its 16 columns of codebook 4 s + g, the constant operand
//               A[i][16 g + b] = (b == i) adds them
// V > 0: up to FEW_FUSED_TOKENS tokens whose index bytes are searched here, by the wave that needs them (sub-vectors of V floats).
template <FewTable T, int TM, int NW, bool XCD, int TC = 1, int V = 0>
__device__ __forceinline__ void gather_few(const FewArgs& a, const Epilogue& ep, const FewSearch& fs = {})
{
    static_assert(TC == 1 || T == FEW_SPARSE, "several column groups: sparse table only");
    static_assert(V == 0 || (T == FEW_SPARSE && TM == 1 && TC == 1), "searched where it is gathered: 16-token items of the sparse table");
    constexpr int UNROLL = V == 8 ? 1 : TC > 1 || V > 0 ? 2 : FEW_UNROLL;  // (registers)
    constexpr int PITCH = T == FEW_ROWS ? FEW_PITCH_ROWS : FEW_PITCH_ONEHOT;
    extern __shared__ __attribute__((aligned(16))) int part[];  // [wave][4 TM registers][PITCH]
    const uint32_t lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // First of the TC column groups (of one tile) and first token.  The grid is (column blocks, token tiles), or, XCD, (8, token tiles, column
    // blocks / 8): XCD p % 8 takes every token tile of the column blocks congruent to it, so that one L2 streams a block's part of the
    // table.  (A form of its own: a test ahead of everything else costs a launch of few tokens 0.2 us, a division as much.)
    uint32_t col_group = blockIdx.x;
    if constexpr (XCD) {
        col_group += 8 * blockIdx.z;
        if (col_group >= a.groups / TC) return;  // whole workgroup, past the last block
    }
    col_group *= TC;
    const uint32_t tok0 = V > 0 ? 0 : blockIdx.y * (16 * TM);
    const uint32_t tile = col_group / a.tile_groups, c = col_group % a.tile_groups;
    const uint32_t op = a.op_groups ? col_group / a.op_groups : 0u;
    const uint32_t wn = 16 * a.tile_groups;
    // 64-token block of the tiled index buffer (16 TM tokens lie in one block), this operator's words
    const uint8_t* ix = a.idx + (size_t)op * ep.op_idx_stride + (size_t)(tok0 / 64) * a.idx_row_bytes * 64 + ((tok0 & 63) + j) * 4;

    v4i acc[TC][TM];
#pragma unroll
    for (int t = 0; t < TC * TM; ++t) acc[t / TM][t % TM] = (v4i){0, 0, 0, 0};

    if constexpr (T != FEW_ROWS) {
        // entry e of column j: ((tile * entries + e) * wn + 16 c + j) * 16 bytes; a K-step is 8 entries
        const int8_t* tab = a.lut + (((size_t)tile * a.steps * 8 + g) * wn + 16 * c + j) * 16;
        ix += T == FEW_SPARSE ? g : (g >> 1) * 256 + (g & 1) * 2;
        for (uint32_t s0 = wave; s0 < a.steps; s0 += NW * UNROLL) {
            v4i lo[UNROLL][TC], hi[UNROLL][TC];
            uint32_t raw[UNROLL][TM];
            constexpr int W = V > 0 ? V : 1;
            float cr[UNROLL][2][W], xr[UNROLL][2][FEW_FUSED_TOKENS][W];  // codebooks 8 s + 4 h + g
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) {
                const uint32_t s = s0 + u * NW;
                if (s < a.steps) {  // uniform
                    if constexpr (V > 0) {
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            const uint32_t cb = 8 * s + 4 * h + g, cbr = cb < fs.CB ? cb : 0;  // (padding: index 0)
                            quad_row<V>(cr[u][h], fs.cent + ((size_t)cbr * fs.C + (j < fs.C ? j : 0)) * V, true);
#pragma unroll
                            for (int t = 0; t < FEW_FUSED_TOKENS; ++t)
                                quad_row<V>(xr[u][h][t], fs.x + (size_t)((uint32_t)t < a.N ? t : 0) * fs.K + cbr * V, fs.aligned);
                        }
                    }
                    const int8_t* p = tab + (size_t)s * 8 * wn * 16;
#pragma unroll
                    for (int e = 0; e < TC; ++e) {
                        lo[u][e] = *reinterpret_cast<const v4i*>(p + e * 256);
                        hi[u][e] = *reinterpret_cast<const v4i*>(p + (size_t)4 * wn * 16 + e * 256);
                    }
#pragma unroll
                    for (int t = 0; t < TM; ++t) {
                        if constexpr (V > 0) continue;
                        else if constexpr (T == FEW_SPARSE) raw[u][t] = ix[(size_t)s * 256 + t * 64];
                        else raw[u][t] = *reinterpret_cast<const uint16_t*>(ix + (size_t)s * 512 + t * 64);
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) {
                if (s0 + u * NW >= a.steps) break;  // uniform
                if constexpr (V > 0) {
                    const uint32_t cb = 8 * (s0 + u * NW), real = fs.CB > cb ? fs.CB - cb : 0;
                    uint32_t word[FEW_FUSED_TOKENS];
#pragma unroll
                    for (int t = 0; t < FEW_FUSED_TOKENS; ++t)
                        if (t == 0 || (uint32_t)t < a.N)  // uniform
                            word[t] = quad_scan<V, false>(xr[u][0][t], cr[u][0], fs.C, lane, real) |
                                      quad_scan<V, false>(xr[u][1][t], cr[u][1], fs.C, lane, real > 4 ? real - 4 : 0) << 16;
                        else word[t] = 0;
                    raw[u][0] = ((j == 1 ? word[1] : word[0]) >> (8 * g)) & 255u;  // (lanes past the tokens: any)
                }
#pragma unroll
                for (int t = 0; t < TM; ++t) {
                    const uint32_t r = raw[u][t];
                    // centroid k of an entry: value 1 in the first slot of group k / 4, position k % 4
                    auto pos = [](uint32_t k) { return (k & 3u) << (4 * ((k >> 2) & 3u)); };
                    v4i aa;
                    uint32_t pw;
                    if constexpr (T == FEW_SPARSE) {
                        const uint64_t v0 = 1ull << ((r & 0x0Cu) << 2), v1 = 1ull << ((r >> 2) & 0x30u);
                        aa = (v4i){(int)(uint32_t)v0, (int)(uint32_t)(v0 >> 32), (int)(uint32_t)v1, (int)(uint32_t)(v1 >> 32)};
                        pw = pos(r & 15) | pos(r >> 4) << 16;
                    } else {
                        // four centroids of 8, a nibble each: codebooks 2e, 2e + 1 in the low and high half of entry e
                        auto val = [&](int n) { return (int)(1u << ((r >> (4 * n) & 4u) << 2)); };
                        aa = (v4i){val(0), val(1), val(2), val(3)};
                        pw = pos(r & 7) | pos(r >> 4 & 7) << 8 | pos(r >> 8 & 7) << 16 | pos(r >> 12 & 7) << 24;
                    }
#pragma unroll
                    for (int e = 0; e < TC; ++e) {
                        const v4i l = lo[u][e], h = hi[u][e];
                        const v8i bb = {l[0], l[1], l[2], l[3], h[0], h[1], h[2], h[3]};
                        acc[e][t] = __builtin_amdgcn_smfmac_i32_16x16x128_i8(aa, bb, acc[e][t], (int)pw, 0, 0);
                    }
                }
            }
        }
    } else {
        // codebook cb, row r: (((chunk * (CB_pad / 16) + cb / 16) * c_tile + r) * 16 + cb % 16) * 16 bytes
        const int8_t* tab = a.lut + (size_t)col_group * (a.steps / 4) * a.c_tile * 256 + g * 16;
        v4i one = (v4i){0, 0, 0, 0};  // byte j of lane (g, j)
#pragma unroll
        for (int w = 0; w < 4; ++w) one[w] = j / 4 == (uint32_t)w ? 1 << (8 * (j % 4)) : 0;
        ix += g;
        for (uint32_t s0 = wave; s0 < a.steps; s0 += NW * FEW_UNROLL) {
            uint32_t raw[FEW_UNROLL][TM];
            v4i row[FEW_UNROLL][TM];
#pragma unroll
            for (int u = 0; u < FEW_UNROLL; ++u)
                if (s0 + u * NW < a.steps) {
#pragma unroll
                    for (int t = 0; t < TM; ++t)  // (index bytes of tokens past the batch were never written)
                        raw[u][t] = tok0 + 16 * t + j < a.N ? ix[(size_t)(s0 + u * NW) * 256 + t * 64] : 0u;
                }
#pragma unroll
            for (int u = 0; u < FEW_UNROLL; ++u) {
                const uint32_t s = s0 + u * NW;
                if (s < a.steps) {
                    const int8_t* p = tab + (size_t)(s / 4) * a.c_tile * 256 + (s % 4) * 64;
#pragma unroll
                    for (int t = 0; t < TM; ++t) row[u][t] = *reinterpret_cast<const v4i*>(p + (size_t)raw[u][t] * 256);
                }
            }
#pragma unroll
            for (int u = 0; u < FEW_UNROLL; ++u) {
                if (s0 + u * NW >= a.steps) break;
#pragma unroll
                for (int t = 0; t < TM; ++t) acc[0][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(one, row[u][t], acc[0][t], 0, 0, 0);
            }
        }
    }

    // lane (g, j) holds: one-hot forms tokens 4 g + r of column position j, byte adder columns 4 g + r of token j
#pragma unroll
    for (int e = 0; e < TC; ++e) {
        if (e) __syncthreads();  // the exchange of the group before has been read
#pragma unroll
        for (int t = 0; t < TM; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[((size_t)wave * TM * 4 + t * 4 + r) * PITCH + lane] = acc[e][t][r];
        __syncthreads();
        for (uint32_t o = threadIdx.x; o < TM * 256; o += NW * 64) {
            const uint32_t x = o % 16, tok = o / 16;  // column position, token of the item
            const uint32_t reg = tok / 16 * 4 + (T == FEW_ROWS ? x % 4 : tok % 4);
            const uint32_t src = T == FEW_ROWS ? x / 4 * 16 + tok % 16 : (tok % 16) / 4 * 16 + x;
            int32_t sum = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) sum += part[((size_t)w * TM * 4 + reg) * PITCH + src];
            const uint32_t n = tok0 + tok;
            const uint32_t f = T == FEW_SPARSE ? tile * wn + few_column(a.tile_groups, c + e, x) : 16 * col_group + x;
            if (n >= a.N || f >= a.M) continue;
            Epilogue epl = ep;
            if (a.op_groups) epl.scale = ep.op_scales[op];
            const float b = ep.bias ? ep.bias[f] : 0.0f;
            a.out[(size_t)n * a.M + f] = ep.act == PIMDL_ACT_GELU_TANH ? dequant<true>(sum, epl, b) : dequant<false>(sum, epl, b);
            if (a.acc_out) a.acc_out[(size_t)n * a.M + f] = sum;
        }
    }
}

// (a name for each, which says in a profile which of the large kernels it stands in for)
template <int TM, int NW, bool XCD>
__global__ __launch_bounds__(NW * 64) void gather_sparse_few_kernel(FewArgs a, Epilogue ep)
{
    gather_few<FEW_SPARSE, TM, NW, XCD>(a, ep);
}
// One or two tokens: search and gather in one launch.  Every workgroup searches all codebooks for its 16 columns, which is less
// than a second launch: a wave requests the centroids, the rows and its part of the table together, 16 codebooks at a time (v = 8: 8, for
// registers), and turns the winners of its own codebooks into its operands without LDS or a barrier.  So there is one round trip up to 256
// codebooks, 128 at v = 8, two beyond.
template <int V, int NW>
__global__ __launch_bounds__(NW * 64) void gather_sparse_few_fused_kernel(FewArgs a, Epilogue ep, FewSearch fs)
{
    gather_few<FEW_SPARSE, 1, NW, false, 1, V>(a, ep, fs);
}
// Sparse table, TC column groups of a tile per workgroup: the operands made from index bytes serve all of them, and a launch has
// fewer workgroups, each with as many loads in flight.  (16 waves, one or two token groups, and all four groups of a
// 64-column tile were slower or spill: N = 1024, 768 codebooks, M = 768 us 8 waves 12.5, 16 12.6, 4 14.8.)
template <int TM, int NW, bool XCD, int TC>
__global__ __launch_bounds__(NW * 64, 4) void gather_sparse_few_wide_kernel(FewArgs a, Epilogue ep)
{
    gather_few<FEW_SPARSE, TM, NW, XCD, TC>(a, ep);
}
template <int TM, int NW, bool XCD>
__global__ __launch_bounds__(NW * 64) void gather_onehot_few_kernel(FewArgs a, Epilogue ep)
{
    gather_few<FEW_PAIRED, TM, NW, XCD>(a, ep);
}
template <int TM, int NW, bool XCD>
__global__ __launch_bounds__(NW * 64) void gather_i8_few_kernel(FewArgs a, Epilogue ep)
{
    gather_few<FEW_ROWS, TM, NW, XCD>(a, ep);
}

// Bytes of a one-hot table (16 bytes per entry and column), and whether token tiles that share it have to meet in one L2: a table that an L2 of 4 MiB
// holds is read from there by every XCD.
uint64_t few_table_bytes(uint64_t steps, uint64_t groups) { return steps * 8 * groups * 256; }
constexpr uint64_t FEW_TABLE_SHARED = 6u << 20;
// workgroups of the XCD that has the most of them, if an XCD takes every token tile of its column blocks
uint64_t few_fullest(uint64_t blocks, uint64_t tiles) { return (blocks + 7) / 8 * tiles; }
// (evenly enough: the XCD that takes one block more has a CU for each of its workgroups, or at most an eighth more than the average;
// 9 column blocks, N = 3100 10.4 in order, 12.1 by XCD)
bool few_even(uint64_t blocks, uint64_t tiles, uint64_t cus)
{
    return 8 * few_fullest(blocks, tiles) <= cus || 64 * few_fullest(blocks, tiles) <= 9 * blocks * tiles;
}
// workgroups that have a CU of their own each (of exactly as many as CUs the last few share some)
uint64_t few_room(uint64_t cus) { return cus - cus / 16; }

// By XCD where the column blocks do not divide by eight by themselves and several token tiles read the same table:
// us, in order / by XCD, three column groups: 2048 codebooks, M = 2048 N = 256 41.1 / 24.8, 1280 x 1280 N = 512 33.2 / 17.6, 256, M =
// 5120 N = 128 10.6 / 7.7; one column group: 2048 N = 128 32.8 / 26.4, 1280 N = 256 22.9 / 18.8; with a CU for every workgroup where the table is
// more than an L2 holds: 4096 -> 1024 (17 MB) N = 40 9.5 / 5.3, 4096 -> 500 v = 2 (17 MB) N = 64 12.5 / 8.3, N = 192 17.1 / 10.7, 1024 ->
// 1024 v = 2 (8.7 MB) N = 40 4.2 / 3.9; 1024 -> 1024 v = 4 (4.3 MB) N = 40 3.2 / 3.2, 768 -> 1280 (4.0 MB) 3.0 / 3.2.
bool few_by_xcd(const FewArgs& f, uint32_t tm, uint32_t tc, uint32_t cus, bool one_hot)
{
    const uint32_t blocks = f.groups / tc, tiles = (f.N + 16 * tm - 1) / (16 * tm);
    const uint64_t fullest = few_fullest(blocks, tiles);
    const bool even = few_even(blocks, tiles, cus);
    // (two items of 64 tokens: 4096 -> 1024 9.0 / 9.3, 5120 -> 1280 11.3 / 10.6)
    const bool shared = one_hot && (tm < 4 || tiles > 2) && 8 * fullest <= few_room(cus) && few_table_bytes(f.steps, f.groups) > FEW_TABLE_SHARED;
    return tiles > 1 && blocks > 8 && blocks % 8 != 0 && (shared || (even && (tc > 1 || tiles * blocks > cus)));
}

template <FewTable T, int TM, int NW, int TC = 1>
int launch_few_as(Ctx* ctx, const Amm& a, const FewArgs& f, const Epilogue& ep, bool xcd)
{
    constexpr int LDS = few_lds_bytes(NW, TM, T == FEW_ROWS ? FEW_PITCH_ROWS : FEW_PITCH_ONEHOT);
    const uint32_t blocks = f.groups / TC, tiles = (f.N + 16 * TM - 1) / (16 * TM);
    const dim3 grid = xcd ? dim3(8, tiles, (blocks + 7) / 8) : dim3(blocks, tiles);
    auto kern = [xcd] {
        if constexpr (TC > 1) return xcd ? gather_sparse_few_wide_kernel<TM, NW, true, TC> : gather_sparse_few_wide_kernel<TM, NW, false, TC>;
        else if constexpr (T == FEW_SPARSE) return xcd ? gather_sparse_few_kernel<TM, NW, true> : gather_sparse_few_kernel<TM, NW, false>;
        else if constexpr (T == FEW_PAIRED) return xcd ? gather_onehot_few_kernel<TM, NW, true> : gather_onehot_few_kernel<TM, NW, false>;
        else return xcd ? gather_i8_few_kernel<TM, NW, true> : gather_i8_few_kernel<TM, NW, false>;
    }();
    if (int rc = allow_dynamic_lds(ctx, reinterpret_cast<const void*>(kern), LDS, "hipFuncSetAttribute(gather_few)")) return rc;
    static const char* const names[] = {TC > 1 ? "gather_sparse_few_wide_kernel" : "gather_sparse_few_kernel", "gather_onehot_few_kernel", "gather_i8_few_kernel"};
    auto name = [](bool x) {
        if constexpr (TC > 1) return KernelName("%s<%d, %d, %s, %d>", names[T], TM, NW, x ? "true" : "false", TC);
        else return KernelName("%s<%d, %d, %s>", names[T], TM, NW, x ? "true" : "false");
    };
    static const KernelName name_of[2] = {name(false), name(true)};
    name_of[xcd].to(a.last_gather);
    a.note_launch(0, LDS, 16 * TM, NW * 64);
    hipLaunchKernelGGL(kern, grid, dim3(NW * 64), LDS, ctx->stream, f, ep);
    return hip_check(ctx, hipGetLastError(), "gather_few launch");
}

constexpr uint32_t FEW_ROWS_BLOCKS = 75;  // column blocks up to which a byte adder launch is priced by its rounds alone if the L2s hold its table (see few_rows)
// Time of such a launch in rounds of 16-token workgroups, which take their codebooks' time each.  Larger items only where they spare rounds: one
// of up to 32 tokens that fits a round where two of 16 do not, or 64 where every one has a CU and the 16 tokens take four rounds and more
// (3.4 times the time; with column blocks that divide by eight, so that the tiles' rows come from one L2).
double few_rows_rounds(const AmmGeom& g, uint32_t n, uint64_t cus, uint32_t* item)
{
    const uint64_t groups = g.M_pad / 16, rounds = ((n + 15) / 16 * groups + cus - 1) / cus;
    *item = n <= 32 && rounds == 2 && groups <= cus ? 32 : rounds >= 4 && groups % 8 == 0 && (n + 63) / 64 * groups <= cus ? 64 : 16;
    return *item == 64 ? 3.4 : (double)rounds;
}

// Whether a byte adder launch of 33..64 centroids is shorter here than on the large kernel, by the prices of gather_few_wanted and, where the
// column blocks do not divide by eight, by what one XCD has to do: by XCD the fullest one has the rounds of its own 1/8 of the
// CUs, and in order the blocks of `tiles` token tiles meet on an XCD, of whose tables what goes beyond 2.5 MB of its L2 takes 0.5 us per MB; the
// large kernel, in tiles of 128 tokens, takes a fifth longer once its part is more than the L2 of 4 MiB.  us of gather, few / large, blocks x
// codebooks: 8 x 192 N = 512 4.1 / 6.5, N = 1024 5.7 / 6.5; 5 x 768 N = 816 11.5 / 24.6; 31 x 768 (by XCD, two rounds) N = 256 16.4 / 25.8; 26 x 768
// N = 160 21.3 / 25.5; not 38 x 192 (by XCD, three rounds) N = 208 7.4 / 6.3; 33 x 192 (in order) N = 128 10.0 / 6.2; 17 x 384 N = 256 13.4 / 9.6; 33 x
// 384 N = 128 17.3 / 9.6.  Of 1179 launches of 1 .. 75 blocks, 16 .. 1024 codebooks and 16 .. 8192 tokens the kernel that this takes is the shorter one, or
// less than 4 % longer, in 1082 (853 with one price for all and no more than 192 tokens).
bool few_rows64_wanted(const AmmGeom& g, uint32_t n, uint64_t cus)
{
    uint32_t item;
    double rounds = few_rows_rounds(g, n, cus, &item), streamed = 0.0;
    const uint64_t blocks = g.M_pad / 16, tiles = (n + item - 1) / item;
    const double eighth_mb = (double)g.CB_pad * 64 * 16 * 1e-6 * (double)blocks / 8;
    // eighths of the table that an XCD reads of so many token tiles in order
    auto meet = [&](uint64_t t) { return std::min<uint64_t>(t, blocks % 8 == 0 ? 1 : blocks % 4 == 0 ? 2 : blocks % 2 == 0 ? 4 : 8); };
    if (blocks % 8 != 0) {
        if (item == 16 && blocks > 8 && tiles > 1 && tiles * blocks > cus && few_even(blocks, tiles, cus))
            rounds = (double)((8 * few_fullest(blocks, tiles) + cus - 1) / cus);
        else streamed = 0.5 * std::max(0.0, (double)meet(tiles) * eighth_mb - std::max(2.5, eighth_mb));
    }
    const double few = 2.5 + rounds * g.CB_pad * 0.0081 + 0.3 * (rounds - 1) + streamed, large = 2.9 + (g.CB + 15) / 16 * 0.29;
    return few < ((double)meet((n + 127) / 128) * eighth_mb > 4.2 ? 1.2 * large : large);
}

// Beyond, and with tables of more than 64 centroids that no L2 holds, rounds overlap, a CU having two workgroups of eight waves, and
// the table is what a launch waits for: us on items of 16, 32 or 64 tokens x 16 columns, each of which takes its codebooks' time a round (less where
// its last tokens are missing) and its token tile's part of the table from memory.  Such a table is read again for every token tile of a column
// block that comes a round later, or on another XCD: by XCD the tiles run together, and it is read once.  (Up to 32 centroids, whose rows any 16
// tokens read nearly all of, only where the blocks meet on several XCDs.)
// us of gather, blocks x codebooks, items of 16 in order / by XCD / 32 / 64 / the large kernel: 200 centroids 192 x 256 N = 76 45.0 / 24.7 / 37.1 /
// 30.1 / 29.4, 80 x 320 N = 144 29.2 / 19.5 / 26.4 / 24.4 / 23.8, 41 x 1536 N = 148 120 / 57 / 99 / 105 / 100, 134 x 421 N = 52 42.1 / 32.6 / 41.3 / 28.2 / 36.3;
// 128 centroids 17 x 746 N = 409 47.7 / 26.1 / 30.4 / 43.4 / 33.9, 192 x 128 N = 43 10.3 / 10.2 / 9.3 / 9.9 / 10.8; 64 centroids 192 x 48 N = 17 3.0 / 3.4 / 3.1 / - /
// 3.8, 475 x 11 N = 8 2.7 (large 3.8), 334 x 340 N = 20 23.6 / 22.0 / 19.3 / - / 19.5; 24 centroids 512 x 512 N = 17 23.4 / 23.5 / 19.5 / - / 22.8, 320 x 320 N =
// 18 9.7 / 11.0 / 11.2 / - / 13.0.  Of 681 launches of 2 .. 600 tokens that these prices decide (four fifths of them went into the figures) the form that
// is taken is within 5 % of the shortest in 635 and beyond 10 % in 25; by rounds alone 160 are beyond 5 %.
struct FewRows {
    uint32_t item;
    bool by_xcd;
    double us;
};
constexpr double FEW_ROWS_L2 = 3.0;  // MB of a table that an L2 holds beside what else there is
// MB that n tokens read of the table: lines of eight codebooks' pieces of a row
double few_rows_read(const AmmGeom& g, uint32_t n) { return (double)g.CB * g.C * g.M_pad * 1e-6 * (1.0 - exp(-8.0 * n / g.C)); }
// XCDs on which the token tiles of a column block meet in order
uint64_t few_rows_meet(uint64_t blocks, uint64_t tiles)
{
    return std::min<uint64_t>(tiles, blocks % 8 == 0 ? 1 : blocks % 4 == 0 ? 2 : blocks % 2 == 0 ? 4 : 8);
}
bool few_rows_priced(const AmmGeom& g, uint32_t n)
{
    const uint64_t blocks = g.M_pad / 16;
    return blocks > FEW_ROWS_BLOCKS || (g.C_tile > 64 && few_rows_read(g, n) / 8 * (double)few_rows_meet(blocks, (n + 15) / 16) > FEW_ROWS_L2);
}
FewRows few_rows(const AmmGeom& g, uint32_t n, uint64_t cus)
{
    // us of a launch; of a codebook and round with a table that the L2s hold, with one that they don't, and of that by XCD
    const struct { uint32_t item; double base, step, step_mem, step_xcd; } forms[] = {
        {16, 2.4, 6.1e-3, 9.2e-3, 9.2e-3}, {32, 3.0, 21.4e-3, 15.6e-3, 14.3e-3}, {64, 3.5, 29.1e-3, 28.7e-3, 37.3e-3}};
    const uint64_t blocks = g.M_pad / 16;
    const double read = few_rows_read(g, n);
    FewRows best{0, false, 1e300};
    for (const auto& f : forms) {
        if (f.item > 16 && 2 * n <= f.item) break;
        const uint64_t tiles = (n + f.item - 1) / f.item, meet = few_rows_meet(blocks, tiles);
        const bool streams = read / 8 * (double)meet > FEW_ROWS_L2;
        const bool by_xcd = streams && tiles > 1 && blocks > 8 && (blocks % 8 != 0 || (tiles * blocks > cus && g.C_tile > 32));
        const double rounds = (double)(((by_xcd ? 8 * few_fullest(blocks, tiles) : tiles * blocks) + cus - 1) / cus);
        const double once = g.C_tile > 32 && !by_xcd ? (double)meet : 1.0;
        const double filled = (0.66 + 0.34 * n / (double)(tiles * f.item)) * (tiles == 1 && f.item > 16 ? 0.83 : 1.0);
        const double us = f.base + (by_xcd ? 0.55 : 0.0) + g.CB_pad * rounds * (by_xcd ? f.step_xcd : streams ? f.step_mem : f.step) * filled +
                          (streams ? (g.C_tile > 32 ? 0.091 : 0.039) * std::max(0.0, read * once - 20.5) : 0.1 * (rounds - 1));
        if (us < best.us) best = {f.item, by_xcd, us};
    }
    return best;
}
// ... and on the large kernel (gather_rows_kernel.hip), whose workgroups go through their slices of 16 codebooks: alone on a CU, two to a CU, and in
// further rounds; its smallest items, which launches that are in question take.
double large_rows_us(const AmmGeom& g, uint32_t n, uint64_t cus)
{
    const bool one_per_cu = g.C_tile == 256;
    const uint64_t blocks = g.M_pad / 16, items = one_per_cu ? (n + 255) / 256 * blocks : (n + 127) / 128 * (g.C_tile <= 32 ? (blocks + 1) / 2 : blocks);
    const double load = (double)items / (double)(one_per_cu ? cus : 2 * cus);
    const double slice = g.C_tile <= 32 ? 0.255 : g.C_tile == 64 ? 0.26 : g.C_tile == 128 ? 0.332 : 0.613;
    const double second = g.C_tile <= 32 ? 1.35 : g.C_tile == 64 ? 0.52 : g.C_tile == 128 ? 0.436 : 1.06, further = g.C_tile <= 32 ? 0.17 : one_per_cu ? 1.02 : 0.0;
    const double table = (double)g.CB * g.C * g.M_pad * 1e-6;
    return 3.65 + (g.CB + 15) / 16 * (slice + second * std::min(std::max(load - 0.5, 0.0), 0.5) + further * std::max(0.0, load - 1.0)) + 0.084 * std::max(0.0, table - 14.0);
}

// Tokens of an item: 16, 32 or 64.  One-hot tables: as few as leave every workgroup a CU of its own.  A wave then makes operands for fewer tokens, and
// what more workgroups read of the table comes from the L2s.  us of gather, items of 16 / 32 / 64 tokens (workgroups): 3072 -> 768 v = 4 N = 64
// 4.6 (192) / 5.4 (96) / 7.3 (48), N = 128 11.8 (384) / 5.5 (192) / 7.4; 768 -> 768 v = 2 N = 128 4.6 (384) / 4.0 (192) / 4.9; 1024 -> 1024 v = 2
// N = 64 5.0 (264) / 4.5 (132) / 5.6; 4096 -> 500 v = 2 by XCD (33 column blocks, five of them on one XCD) N = 64 8.3 (20 on that XCD) / 10.5 / 15.0, N =
// 100 13.0 (35) / 10.6 (20) / 15.2; 8 centroids 3072 -> 768 N = 64 3.5 / 4.1 / 5.7.
// Byte adder (up to FEW_ROWS_BLOCKS), whose tokens' rows are read whatever the item: 32 centroids 3072 -> 768 N = 64 8.6 / 15.0 / 17.3, N = 100 14.8 (336) / 15.0 / 17.6, 3072
// -> 3072 N = 32 19.5 (384) / 15.2; 100 centroids 768 -> 2304 N = 32 9.3 (288) / 7.8; 64 centroids 3072 -> 768 v = 8 N = 64 5.4 / 9.3 / 9.4; 200
// 768 -> 768 N = 256 10.5 (768) / - / 11.2 (192), N = 300 13.0 (912) / - / 10.7 (240).
uint32_t few_item(const AmmGeom& g, uint32_t n, uint64_t cus)
{
    const uint64_t groups = g.M_pad / 16;
    if (g.gather_kind == 0) {
        uint32_t item;
        few_rows_rounds(g, n, cus, &item);
        return item;
    }
    const uint64_t table = (uint64_t)g.CB_pad * g.C_tile * g.M_pad;
    for (uint32_t item = 16; item < 64; item *= 2) {
        const uint64_t tiles = (n + item - 1) / item;
        const bool by_xcd = groups % 8 != 0 && table > FEW_TABLE_SHARED;  // (few_by_xcd)
        if (tiles == 1 || (by_xcd ? 8 * few_fullest(groups, tiles) : tiles * groups) <= few_room(cus)) return item;
    }
    return 64;
}

// Sixteen waves while every workgroup has a CU to itself, eight (two workgroups share a CU) beyond: us at 3072 -> 768,
// 16 centroids, sixteen / eight waves: N = 64 7.5 / 8.4 (48 workgroups), N = 512 14.1 / 13.1 (384 workgroups).
template <FewTable T>
int launch_few(Ctx* ctx, const Amm& a, const FewArgs& f, const Epilogue& ep)
{
    const uint32_t cus = ctx->prop.multiProcessorCount;
    uint32_t item;
    bool xcd;
    if (T == FEW_ROWS && few_rows_priced(a.g, f.N)) {
        const FewRows r = few_rows(a.g, f.N, cus);
        item = r.item;
        xcd = r.by_xcd;
    } else {
        item = few_item(a.g, f.N, cus);
        xcd = few_by_xcd(f, item / 16, 1, cus, T != FEW_ROWS);
    }
    const bool deep = f.groups * ((f.N + item - 1) / item) <= cus;
    if (item == 16) return deep ? launch_few_as<T, 1, 16>(ctx, a, f, ep, xcd) : launch_few_as<T, 1, 8>(ctx, a, f, ep, xcd);
    if (item == 32) return deep ? launch_few_as<T, 2, 16>(ctx, a, f, ep, xcd) : launch_few_as<T, 2, 8>(ctx, a, f, ep, xcd);
    return deep ? launch_few_as<T, 4, 16>(ctx, a, f, ep, xcd) : launch_few_as<T, 4, 8>(ctx, a, f, ep, xcd);
}

// fp32 tables (and int8 ones with a scale per group of codebooks, resident as floats): a lane is one column of one
// token and adds its entries in ascending codebook order -- the order, and so the bits, of gather_f32_kernel -- with the
// loads of two times 32 codebooks in flight.  The table is read where it lies: every entry that is added is fetched, and
// nothing else.
template <int FB, int IDX_BITS, bool GROUPED>
__global__ __launch_bounds__(64) void gather_f32_few_kernel(const uint8_t* __restrict__ idx, const float* __restrict__ lut,
                                                            float* __restrict__ out, uint32_t N, uint32_t M, uint32_t CB_pad,
                                                            uint32_t idx_row_bytes, const float* __restrict__ bias,
                                                            const float* __restrict__ scales, uint32_t CB, uint32_t group,
                                                            uint32_t act, uint32_t colblocks, uint32_t c_tile, uint32_t piece)
{
    constexpr int TOK = 64 / FB, WORDS = IDX_BITS;  // tokens per wave; index words of 32 codebooks
    const uint32_t colblk = blockIdx.x % colblocks, e = threadIdx.x % FB;
    const uint32_t tok = blockIdx.x / colblocks * TOK + threadIdx.x / FB, f = colblk * FB + e;
    const uint32_t* ix = reinterpret_cast<const uint32_t*>(idx + (size_t)(tok < N ? tok : N - 1) * idx_row_bytes);
    // entry of row r: [row][FB], or [FB / piece][row][piece]
    const uint32_t row = piece ? piece : FB;
    const float* tab = lut + (size_t)colblk * CB_pad * c_tile * FB + (piece ? e / piece * c_tile * piece + e % piece : e);
    const uint32_t per_cb = c_tile * FB, batches = CB_pad / 32;

    uint32_t w[WORDS];
    float v[2][32];
    auto load_ix = [&](uint32_t b) {
#pragma unroll
        for (int i = 0; i < WORDS; ++i) w[i] = ix[(b < batches ? b : batches - 1) * WORDS + i];
    };
    auto fetch = [&](uint32_t b, float (&dst)[32]) {
        const float* p = tab + (size_t)b * 32 * per_cb;
#pragma unroll
        for (int k = 0; k < 32; ++k) {
            constexpr int PER = 32 / IDX_BITS;
            dst[k] = p[k * per_cb + (w[k / PER] >> (k % PER * IDX_BITS) & ((1u << IDX_BITS) - 1)) * row];
        }
    };
    float acc = 0.0f, tot = 0.0f;
    uint32_t cb = 0, in_group = 0, gi = 0;
    auto add = [&](const float (&src)[32]) {
#pragma unroll
        for (int k = 0; k < 32; ++k) {
            acc = __fadd_rn(acc, src[k]);
            if constexpr (GROUPED) {
                // codebooks past CB are padding (zero rows) and belong to no group
                if (cb < CB && (++in_group == group || cb + 1 == CB)) {
                    tot = __fadd_rn(tot, __fmul_rn(acc, scales[gi++]));
                    acc = 0.0f;
                    in_group = 0;
                }
                ++cb;
            }
        }
    };
    load_ix(0);
    fetch(0, v[0]);
    load_ix(1);
    for (uint32_t b = 0; b < batches; b += 2) {
        if (b + 1 < batches) fetch(b + 1, v[1]);
        load_ix(b + 2);
        add(v[0]);
        if (b + 1 < batches) {
            if (b + 2 < batches) fetch(b + 2, v[0]);
            load_ix(b + 3);
            add(v[1]);
        }
    }
    if (tok < N && f < M) out[(size_t)tok * M + f] = activate(__fadd_rn(GROUPED ? tot : acc, bias ? bias[f] : 0.0f), act);
}

template <int FB, int IDX_BITS, bool GROUPED>
int launch_f32_few(Ctx* ctx, const Amm& a, const uint8_t* d_idx, float* d_out, uint32_t n)
{
    const AmmGeom& g = a.g;
    const uint32_t colblocks = g.M_pad / FB, tok = 64 / FB;
    static const KernelName name("gather_f32_few_kernel<%d, %d, %s>", FB, IDX_BITS, GROUPED ? "true" : "false");
    name.to(a.last_gather);
    a.note_launch(0, 0, tok, 64);
    hipLaunchKernelGGL((gather_f32_few_kernel<FB, IDX_BITS, GROUPED>), dim3(colblocks * ((n + tok - 1) / tok)), dim3(64), 0, ctx->stream,
                       d_idx, reinterpret_cast<const float*>(a.d_lut), d_out, n, g.M, g.CB_pad, g.idx_row_bytes, a.d_bias,
                       a.d_scales, g.CB, a.desc.scale_group, a.desc.activation, colblocks, g.C_tile, g.lut_chunk);
    return hip_check(ctx, hipGetLastError(), "gather_f32_few_kernel launch");
}

}  // namespace

// Column groups that a workgroup of a launch on the sparse kernel's table takes (0: the large kernel is the shorter launch): as few as leave
// every workgroup a CU of its own.  us, large / one group / several, N tokens: 768 codebooks, M = 768 N = 512 19.1 / 12.6 / 12.1 (three), 1024 19.3 /
// 17.7 / 12.6, 2048 19.7 / 30.9 / 20.0; 1024, M = 1024 N = 512 26.0 / 16.8 / 12.0 (two), 700 27 / 24 / 20; 2048, M = 2048 N = 400 53 / 51 / 35 (two);
// 192, M = 3072 N = 256 8.1 / 8.1 / 6.7 (three), 512 8.6 / 13.5 / 9.3; 384, M = 1280 N = 256 11.9 / 8.0 / 8.3 (three), 400 12.8 / 11.2 / 8.6; 256, M =
// 4096 N = 128 9.5 / 7.8 / 6.5 (two), 200 10.8 / 11.7 / 9.2; 96-column tiles 192, M = 2304 N = 256 11.7 / 9.1 / 7.3 (three), 400 12.5 / 11.2 / 8.3 (two).
// One token tile (the large kernel's chain is the same for one token): 512, M = 8192 N = 1 17.6 / 12.6, 32 18.2 / 12.7, 64 18.3 /
// 14.4 / 14.2 (three); 192, M = 8192 N = 1 8.2 / 3.8, M = 12000 9.8 / 6.2, N = 64 10.7 / 9.3 / 8.8 (three).
uint32_t few_column_groups(const Ctx* ctx, const AmmGeom& g, uint32_t n)
{
    const uint64_t cus = ctx->prop.multiProcessorCount, groups = g.M_pad / 16, item = few_item(g, n, cus), tiles = (n + item - 1) / item;
    const uint64_t wgs = tiles * groups;
    if (wgs <= cus) return 1;
    if (n <= 32) return wgs <= 4 * cus ? 1 : 0;
    const uint32_t tc = g.q % 2 == 0 && (wgs / 2 <= cus || g.q % 3 != 0) ? 2 : 3;
    const uint64_t wide = wgs / tc;
    if (g.q == 3) return wgs <= 2 * cus ? (g.CB_pad >= 640 ? 3 : 1) : wide <= cus ? 3 : 0;
    return wide <= cus || (wide <= 2 * cus && g.CB_pad >= 128) ? tc : wgs <= 2 * cus ? 1 : 0;
}

// Whether these kernels are the shorter launch.  The large kernels' time is flat while their items do not fill the chip
// (us, large / few): one-hot tables 768 -> 3072 8.1 / 3.0 at N = 1, 8.7 / 4.1 at 64, 9.1 / 9.7 at 300; 3072 -> 768
// 19.8 / 4.5 at 1, 20.2 / 7.7 at 150, 19.8 / 13.1 at 512, 20.3 / 18.2 at 1024; 8 centroids 3072 -> 768 15.4 / 5.9 at 64,
// 15.6 / 10.0 at 512: up to two workgroups of this launch per CU (the paired table; for the sparse one few_column_groups decides).
// The byte adder and the floats read every gathered piece from the caches on its own, which costs in proportion to
// tokens x codebooks x columns -- the byte adder by rounds of workgroups of 16 tokens x 16 columns, which take their codebooks' time each (see few_rows) --;
// against that stands the large kernels' chain of slices.  Byte adder, 3072 -> 768, 32 centroids: 17.6 / 4.4 at N = 1, 17.4 / 8.6 at 64,
// 17.6 / 14.8 at 128 (384 workgroups), 17.8 / 20.9 at 192; 768 -> 768 6.8 / 3.8 at 70, 7.0 / 5.4 at 150, 7.2 / 8.6 at 300; 768 -> 3072 8.3 / 5.4 at
// 32, 8.8 / 10.9 at 100; 16 codebooks, M = 1040 3.3 / 2.6 at 32, 3.8 / 4.2 at 300; 64 centroids 1024 -> 1024 7.2 / 4.4 at 50, 7.4 / 6.6 at 100, 7.6 / 8.9 at
// 150; 4096 -> 512 27.8 / 12.8 at 64, 31.2 / 20.7 at 192; 128 centroids 768 -> 768 7.4 / 4.3 at 70, 7.6 / 8.3 at 200; 200 centroids 1000 -> 1001 15.7 /
// 6.8 at 32, 16.0 / 12.3 at 150, 19.2 / 21.9 at 400.  Floats, 16 centroids (the large kernel with 64-token workgroups): 3072 -> 768 23.7 / 14.4 at 1,
// 24.0 / 19.6 at 13, 25.5 / 28.7 at 64; 768 -> 3072 8.6 / 5.2 at 1, 8.4 / 9.3 at 13; 32 centroids 3072 -> 768 44 / 33 at 1,
// 47 / 71 at 64; 200 centroids (whole rows) 1000 -> 1001 49 / 5.3 at 1, 51 / 32 at 64, 56 / 73 at 150; a scale per 5
// codebooks 19.8 / 18.7 at 1, 19.7 / 22.6 at 13; 64 centroids (large / few; a piece costs more where the caches do not hold the
// table), 96 codebooks, M = 2441 16.2 / 10.2 at 32, 16.5 / 24.3 at 93; M = 554 15.7 / 9.1 at 150, 17.5 / 17.2 at 400; 768 codebooks,
// M = 2441 122 / 63 at 32, 123 / 183 at 93; a scale per 8 codebooks, M = 1001 25 / 31 at 283.  The estimates are fits to these.
bool gather_few_wanted(const Ctx* ctx, const Amm& a, uint32_t n)
{
    const AmmGeom& g = a.g;
    if (g.tune_token_item || g.tune_cb_per_slice || g.tune_xcd_col_split) return false;  // settings of the large kernels
    const uint64_t cus = ctx->prop.multiProcessorCount, item = few_item(g, n, cus), wgs = (n + item - 1) / item * (g.M_pad / 16);
    const double pieces = (double)n * g.CB_pad * (g.M_pad / 16);  // of 16 columns
    if (a.desc.lut_dtype == PIMDL_LUT_F32 || a.grouped) {
        const bool bounds = a.grouped && !a.prescaled;  // a scale to apply at the end of every group
        if (g.lut_chunk) return pieces * (g.lut_chunk == 2 ? 18e-6 : 7.5e-6) < (bounds ? 1.0 : 1.4 + 0.0103 * g.CB_pad);
        const double piece = g.q != 4 ? 32e-6 : bounds || a.lut_bytes > (48u << 20) ? 6.5e-6 : 5e-6;
        return 2.7 + g.CB_pad * (bounds ? 0.062 : 0.0137) + pieces * piece < 4.0 + g.CB_pad * (bounds ? 0.14 : 0.07);
    }
    if (g.gather_kind == 0) {
        if (few_rows_priced(g, n)) return g.idx_bits == 8 && few_rows(g, n, cus).us < large_rows_us(g, n, cus);
        if (g.C_tile == 64) return g.idx_bits == 8 && few_rows64_wanted(g, n, cus);
        const uint64_t slices = (g.CB + 15) / 16;
        uint32_t rows_item;
        const double rounds = few_rows_rounds(g, n, cus, &rows_item);
        const double few = 2.5 + rounds * g.CB_pad * (g.C_tile < 64 ? 0.0081 : g.C_tile == 128 ? 0.014 : 0.0125) + 0.3 * (rounds - 1);
        return g.idx_bits == 8 && few < 3.3 + (double)slices * (0.2 + 0.003 * g.C_tile);
    }
    if (g.gather_kind == 2 ? g.C_tile == 32 : g.C_tile != 8) return false;  // tables only a tuning asks for
    return g.gather_kind == 2 ? few_column_groups(ctx, g, n) != 0 : wgs <= 2 * cus;
}

// Whether one launch searches and gathers: up to 256 (token, codebook) pairs, which the 16 waves of every workgroup search side by side.
// us a pass, two launches / one, launched one by one (replayed from a graph): 192 codebooks, v = 4, M = 3072 N = 1
// 6.8 / 4.5 (4.9 / 4.2), N = 2 6.9 / 5.4 (4.8 / 5.1); 96 codebooks, v = 8, M = 2304 N = 1 7.1 / 3.9 (4.4 / 3.7), N = 2 7.1 / 4.6 (4.6 / 4.2); 25
// codebooks 6.9 / 4.0 (4.1 / 2.6); 384 codebooks, v = 2, M = 768 N = 1 7.0 / 6.2 (5.4 / 5.8); 512, v = 4 6.8 / 7.7 (6.0 / 7.5).  Nor with more
// workgroups than CUs, each of which would search again: 256, v = 4, M = 4096 6.2 / 8.3 (5.6 / 8.2), 128, v = 8 6.3 / 6.3 (4.8 / 6.1).
// At the line, 256 workgroups: 192 codebooks, v = 4 8.1 / 4.7 (5.1 / 4.5), 256 8.1 / 5.8 (5.3 / 5.3); 256, v = 2 8.2 / 5.8 (5.3 / 5.3).  v = 8,
// whose second round trip begins beyond 128 codebooks, M = 2304: 128 6.8 / 4.7 (4.7 / 4.2), 160 7.0 / 5.0 (4.9 / 4.6), 192 7.0 / 5.6 (5.0 / 4.9), 224 6.7 /
// 6.1 (5.2 / 5.5), 256 7.9 / 6.5 (5.3 / 5.9): what a program that launches one by one gains there outweighs what a graph loses.
bool amm_few_wanted(const Ctx* ctx, const Amm& a, uint32_t n)
{
    const AmmGeom& g = a.g;
    return n <= FEW_FUSED_TOKENS && n * g.CB_pad <= 256 && a.desc.lut_dtype == PIMDL_LUT_I8 && !a.grouped && g.gather_kind == 2 && g.C <= 16 &&
           (g.v == 2 || g.v == 4 || g.v == 8) && !g.tune_search && !g.tune_search_tile && !ccs_exact_only() && !ccs_f32_only() &&
           g.M_pad / 16 <= (uint32_t)ctx->prop.multiProcessorCount && gather_few_wanted(ctx, a, n);
}

int launch_amm_few(Ctx* ctx, const Amm& a, const float* d_x, float* d_out, uint32_t n, float scale, float lut_bias_term)
{
    const AmmGeom& g = a.g;
    constexpr int NW = 16, LDS = few_lds_bytes(NW, 1, FEW_PITCH_ONEHOT);
    Epilogue ep = {};
    ep.scale = scale;
    ep.lut_bias_term = lut_bias_term;
    ep.bias = a.d_bias;
    ep.act = a.desc.activation;
    const FewArgs f = {nullptr, reinterpret_cast<const int8_t*>(a.d_lut), d_out, nullptr, n, g.M, g.M_pad / 16, g.CB_pad / 8, g.q, g.C_tile,
                       g.idx_row_bytes, 0};
    const FewSearch fs = {d_x, a.d_centroids, g.K, g.CB, g.C, (reinterpret_cast<uintptr_t>(d_x) & 15) == 0};
    auto kern = g.v == 2 ? gather_sparse_few_fused_kernel<2, NW> : g.v == 4 ? gather_sparse_few_fused_kernel<4, NW> : gather_sparse_few_fused_kernel<8, NW>;
    if (int rc = allow_dynamic_lds(ctx, reinterpret_cast<const void*>(kern), LDS, "hipFuncSetAttribute(gather_few_fused)")) return rc;
    static const KernelName names[] = {KernelName("gather_sparse_few_fused_kernel<2, %d>", NW), KernelName("gather_sparse_few_fused_kernel<4, %d>", NW),
                                       KernelName("gather_sparse_few_fused_kernel<8, %d>", NW)};
    names[g.v / 4].to(a.last_gather);
    a.note_launch(0, LDS, 16, NW * 64);
    hipLaunchKernelGGL(kern, dim3(f.groups), dim3(NW * 64), LDS, ctx->stream, f, ep, fs);
    return hip_check(ctx, hipGetLastError(), "gather_few_fused launch");
}

int launch_gather_few(Ctx* ctx, const Amm& a, const uint8_t* d_idx, float* d_out, int32_t* d_acc, uint32_t n, float scale,
                      float lut_bias_term)
{
    const AmmGeom& g = a.g;
    if (a.desc.lut_dtype == PIMDL_LUT_F32 || a.grouped) {
        if (a.grouped && !a.prescaled) {
            if (g.idx_bits == 4) return launch_f32_few<16, 4, true>(ctx, a, d_idx, d_out, n);
            if (g.q == 4) return launch_f32_few<16, 8, true>(ctx, a, d_idx, d_out, n);
            return launch_f32_few<8, 8, true>(ctx, a, d_idx, d_out, n);
        }
        if (g.idx_bits == 4) return launch_f32_few<16, 4, false>(ctx, a, d_idx, d_out, n);
        if (g.q == 4) return launch_f32_few<16, 8, false>(ctx, a, d_idx, d_out, n);
        return launch_f32_few<8, 8, false>(ctx, a, d_idx, d_out, n);
    }
    Epilogue ep;
    ep.scale = scale;
    ep.lut_bias_term = lut_bias_term;
    ep.bias = a.d_bias;
    ep.act = a.desc.activation;
    ep.op_scales = a.d_op_scales;
    ep.op_col_tiles = a.op_col_tiles;
    ep.op_idx_stride = a.op_idx_stride;
    FewArgs f = {d_idx, reinterpret_cast<const int8_t*>(a.d_lut), d_out, d_acc, n, g.M, g.M_pad / 16, 0, g.q, g.C_tile,
                 g.idx_row_bytes, a.op_col_tiles * g.q};
    if (g.gather_kind == 2) {
        f.steps = g.CB_pad / 8;
        switch (few_column_groups(ctx, g, n)) {
            case 2: return launch_few_as<FEW_SPARSE, 4, 8, 2>(ctx, a, f, ep, few_by_xcd(f, 4, 2, ctx->prop.multiProcessorCount, true));
            case 3: return launch_few_as<FEW_SPARSE, 4, 8, 3>(ctx, a, f, ep, few_by_xcd(f, 4, 3, ctx->prop.multiProcessorCount, true));
        }
        return launch_few<FEW_SPARSE>(ctx, a, f, ep);
    }
    if (g.gather_kind == 1) {
        f.steps = g.CB_pad / 16;
        return launch_few<FEW_PAIRED>(ctx, a, f, ep);
    }
    f.steps = g.CB_pad / 4;
    f.tile_groups = 1;
    return launch_few<FEW_ROWS>(ctx, a, f, ep);
}

}  // namespace pimdl
