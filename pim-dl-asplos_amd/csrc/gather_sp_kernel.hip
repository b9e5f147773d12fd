// LUT gather-accumulate on the sparse matrix instruction (gfx950), int8 tables with up to 32 centroids
// (9..32 always; up to 8 where the launch rule of plan_geometry prefers it to the paired dense kernel).
//
// Same operator as the other gather kernels (inference-engine/src/dpu/pim_lut_kernel.c:97-2296, row-major
// statement inference-engine/test/test_amm.cpp:164-175, epilogue inference-engine/src/host/pim_lut_host.cpp:190-203):
//     acc[n][f] = sum over cb of lut[cb][idx[n][cb]][f]          (int8 table, int32 sum, exact)
// in the reference's own matrix form (model-calibration/LUTNeuro/LUTLinear_t.py:78, bmm(one_hot, lut)).
//
// A one-hot row over the 16 centroids of a codebook has at most one non-zero in every group of four
// positions, which is a valid 2:4 structured-sparse operand.  v_smfmac_i32_16x16x128_i8 multiplies a
// 16 x 128 matrix given in that compressed form (per lane: 16 value bytes + 16 two-bit positions) by a dense
// 128 x 16 one: with the one-hot as the sparse operand, ONE instruction gathers and adds 8 codebooks for
// 16 tokens x 16 columns, twice what the dense v_mfma_i32_16x16x64_i8 form of the one-hot product does, at
// the same issue rate (measured: 16.5 clocks per instruction and SIMD for either).
//
// Operands of one instruction (K-step = 8 codebooks b = 0..7 of a slice), lane l = 16 g + i:
//   sparse A (tokens x K)  lane (g, i) holds, for token i of the 16-token group, codebooks 2g (value bytes
//             0..7) and 2g+1 (value bytes 8..15): each codebook is four groups of two value slots; the group
//             that contains the token's centroid c (group c / 4) has value 1 in its first slot with position
//             c % 4, everything else is 0.  Both codebooks' nibbles are one byte of the packed index row.
//             The 8 value bytes of a nibble are the 64-bit number 1 << 16 (c / 4): one shift.  (With 17..32
//             centroids they come from a table in LDS, entry c 16 bytes apart: 8-byte reads of such entries do
//             not meet in a bank.)  The lane's whole position word (16 bits per nibble) comes from a second
//             table with one 4-byte word per value of the index byte.
//   dense B (K x columns)  lane (g, j) holds column j's 16 centroid entries of codebook g (bytes 0..15) and
//             of codebook g + 4 (bytes 16..31): two 16-byte reads of the tiled table, whose layout is that
//             of the dense one-hot kernel ([column tile][codebook][column][16 centroids]).
//   D (tokens x columns)   lane (g, j) holds tokens 4g..4g+3 of the group for column j.
// (This pairing of lane groups and codebooks was read off the instruction on the device with one-hot probes.)
//
// A lane thus ends up with four tokens of ONE column per 16-column group.  So that its stores are still
// 16 bytes wide, the columns of a tile are dealt to the 16-column groups in pieces: the first 4 * (TN / 4)
// groups in fours (group c of a four holds columns 4 j + c: a lane's four accumulator tiles are four
// consecutive columns), then a pair (columns 2 j + c), then a single group.  The permutation is applied once
// when the table is tiled at upload (sparse_tile_column); reads of the table from LDS stay consecutive.
//
// Work decomposition, staging through LDS with global_load_lds, the dealing of items to the XCDs, the fused
// de-quantisation / bias / GELU epilogue and operator groups are those of the dense one-hot kernel.
//
// 17..32 centroids (WIDE): a codebook of 32 centroids is two of 16 side by side, of which the token's centroid
// lies in one and the other contributes nothing.  The table is tiled as 2 CB codebooks of 16 (centroids 0..15,
// then 16..31), the index row holds one byte per codebook where the 16-centroid form holds two nibbles, and the
// lane looks its byte up in two 32-entry tables: the first has the one-hot entries for bytes 0..15 and zero
// entries for 16..31, the second the other way round.  Everything else is the same kernel; one instruction then
// covers 4 codebooks.
#include "gather_common.h"

namespace pimdl {

// column (within its tile of 16 * tn columns) stored at position s = 16 c + j of the tile
uint32_t sparse_tile_column(uint32_t tn, uint32_t s)
{
    const uint32_t c = s / 16, j = s % 16;
    const uint32_t n4 = tn / 4 * 4;                 // groups dealt in fours
    const uint32_t n2 = n4 + (tn % 4) / 2 * 2;      // ... then a pair
    if (c < n4) return 16 * (c / 4 * 4) + 4 * j + c % 4;
    if (c < n2) return 16 * n4 + 2 * j + (c - n4);
    return 16 * c + j;
}

namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v2i __attribute__((ext_vector_type(2)));

// Waves per workgroup (NW): 4, two or three workgroups per CU -- or 8, one workgroup per CU: two waves per
// SIMD, but a LUT slice is copied into LDS once for 512 tokens instead of 256 and the CU's whole LDS belongs
// to one workgroup (slices twice as deep, half as many barriers).
constexpr int sp_tok_item(int tm, int nw = 4) { return nw * tm * 16; }
// Workgroups per CU: 48- and 64-column tiles of 64 tokens per wave fit 168 registers, and with slices of 16 codebooks (64 columns: in two
// buffers) three workgroups fit a CU.  The third wave of a SIMD runs where the other two wait for operands, slices or stores: three
// operators, inputs and outputs taking turns, two against three, us a pass: 768 -> 3072 N = 8192 57.1 / 56.2, N = 12608 85.1 / 80.9; 1024 -> 4096 N = 32768
// 319 / 308.  (Eight waves of 32 tokens each, two such workgroups per CU -- four waves per SIMD -- are slower: a wave then re-reads every
// table entry for two token groups instead of four.  Four workgroups of 48 columns on 128 registers spill: 60 -> 77 us.  Position
// words from vector operations instead of the table in LDS: 79 -> 88 us at 768 -> 3072, N = 12608.)
constexpr bool sp_three_per_cu(int tn, int tm, int gs, int nw, bool wide) { return nw == 4 && tm == 4 && gs == 16 && tn <= 4 && !wide; }
constexpr int sp_wgs_per_cu(int tn, int tm, int gs, int nw, bool wide)
{
    return nw != 4 ? 1 : sp_three_per_cu(tn, tm, gs, nw, wide) ? 3 : 2;
}
// 64-token index blocks a workgroup keeps per slice: a wave of 32 tokens shares its block with its neighbour (both
// copy the same bytes to the same place)
constexpr int sp_ix_blocks(int tm, int nw) { return nw * tm * 16 / 64; }
constexpr int sp_nbuf(int tn, int tm, int gs, int nw, bool wide) { return gs > 16 || (tn == 4 && sp_three_per_cu(tn, tm, gs, nw, wide)) ? 2 : 3; }
// value tables (17..32 centroids only: two tables of 32 entries of 16 bytes); then the position words, one per index byte
constexpr int sp_value_table_bytes(bool wide) { return wide ? 1024 : 0; }
constexpr int sp_table_bytes(bool wide) { return sp_value_table_bytes(wide) + 1024; }
// ks: waves that share a token block and split the codebooks of a slice between them (1 or 2)
constexpr int sp_lds_bytes(int tn, int tm, int gs, int nw, bool wide, int ks = 1)
{
    return sp_table_bytes(wide) + sp_nbuf(tn, tm, gs, nw, wide) * (gs * 16 * tn * 16 + sp_ix_blocks(tm, nw / ks) * 64 * 4 * (gs / 8));
}

template <int OFF>
__device__ __forceinline__ void lds_read64(v2i& dst, uint32_t addr)
{
    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}
template <int OFF>
__device__ __forceinline__ void lds_read32(int& dst, uint32_t addr)
{
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}
template <int N>
__device__ __forceinline__ void lgkm_wait()
{
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N < 15 ? N : 15) : "memory");
}

// a pointer that is the same in every lane, moved to scalar registers
template <class T>
__device__ __forceinline__ T* uniform_ptr(T* p)
{
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return reinterpret_cast<T*>(((uint64_t)hi << 32) | lo);
}

// CB_pad: codebooks of 16 centroids in the tiled table (twice the operator's for WIDE)
// KS = 2 (eight waves): waves w and w + 4 hold the same 64 tokens and take one half of every slice's codebooks each;
// the halves are added through LDS before the epilogue.  An item is then 256 tokens: a launch too small to give
// every CU a 512-token item still fills the chip with TM = 4 tiles and copies a slice once per 256 tokens.
// The body of both kernels is gather_sp_body.h: a shared function compiles to other code than the kernel alone.
template <int TN, int TM, int GS, int NW, bool WIDE, int KS = 1>
__global__ __launch_bounds__(NW * 64, sp_wgs_per_cu(TN, TM, GS, NW, WIDE) * NW / 4 /* waves per SIMD */) void gather_sparse_kernel(
    const uint8_t* __restrict__ idx, const int8_t* __restrict__ lut, float* __restrict__ out,
    int32_t* __restrict__ acc_out, uint32_t N, uint32_t M, uint32_t CB_pad, uint32_t idx_row_bytes,
    uint32_t n_token_tiles, uint32_t n_items, Epilogue ep, XcdMap xmap)
{
    constexpr bool STREAM = true;
#include "gather_sp_body.h"
}
// the launch deals its items in blocks of token tiles
template <int TN, int TM, int GS, int NW>
__global__ __launch_bounds__(NW * 64, sp_wgs_per_cu(TN, TM, GS, NW, false) * NW / 4) void gather_sparse_blocks_kernel(
    const uint8_t* __restrict__ idx, const int8_t* __restrict__ lut, float* __restrict__ out,
    int32_t* __restrict__ acc_out, uint32_t N, uint32_t M, uint32_t CB_pad, uint32_t idx_row_bytes,
    uint32_t n_token_tiles, uint32_t n_items, Epilogue ep, XcdBlocks xmap)
{
    constexpr bool WIDE = false;
    constexpr int KS = 1;
    constexpr bool STREAM = true;
#include "gather_sp_body.h"
}
// The same two for rows that are written with plain stores (see streaming_stores): another type of the last argument, so that
// the code of the others stays what it is without a second epilogue (which cost a forward of 48-column tiles 0.6 %).
template <class Map>
struct PlainStores : Map {};
template <int TN, int TM, int GS, int NW, bool WIDE, int KS = 1>
__global__ __launch_bounds__(NW * 64, sp_wgs_per_cu(TN, TM, GS, NW, WIDE) * NW / 4 /* waves per SIMD */) void gather_sparse_kernel(
    const uint8_t* __restrict__ idx, const int8_t* __restrict__ lut, float* __restrict__ out,
    int32_t* __restrict__ acc_out, uint32_t N, uint32_t M, uint32_t CB_pad, uint32_t idx_row_bytes,
    uint32_t n_token_tiles, uint32_t n_items, Epilogue ep, PlainStores<XcdMap> xmap)
{
    constexpr bool STREAM = false;
#include "gather_sp_body.h"
}
template <int TN, int TM, int GS, int NW>
__global__ __launch_bounds__(NW * 64, sp_wgs_per_cu(TN, TM, GS, NW, false) * NW / 4) void gather_sparse_blocks_kernel(
    const uint8_t* __restrict__ idx, const int8_t* __restrict__ lut, float* __restrict__ out,
    int32_t* __restrict__ acc_out, uint32_t N, uint32_t M, uint32_t CB_pad, uint32_t idx_row_bytes,
    uint32_t n_token_tiles, uint32_t n_items, Epilogue ep, PlainStores<XcdBlocks> xmap)
{
    constexpr bool WIDE = false;
    constexpr int KS = 1;
    constexpr bool STREAM = false;
#include "gather_sp_body.h"
}

// Streaming stores where rows are whole half lines of 64 bytes.  Where they are not, a row's part of a tile ends inside one that the neighbour
// tile writes the rest of: streamed, the two parts go to memory one by one; plain stores meet in L2.  They also push the table out of it, so
// that one of about an L2 of 4 MiB, or an output that shows nothing of all this, is better off streamed.  Widths that four does not
// divide (16 bytes at any multiple of four bytes, where they used to be four stores of one column each) are plain always.  us a pass,
// inputs and outputs in turn, streamed / plain: 11 codebooks, M = 1112 N = 16034 47.2 / 25.4, 64 N = 13893 38.1 / 27.3, 256 (4.5 MB) N = 10225 52.3 /
// 58.2; 192 codebooks, M = 1244 N = 7696 41.6 / 34.6, 2340 (7.2 MB) N = 19245 106.8 / 113.0; 326, 744 (4.2 MB) N = 20054 113.3 / 117.8; 64, M = 828 N =
// 3989 (13 MB of output) 13.2 / 14.2; half lines, 20 codebooks, M = 624 N = 15729 20.5 / 21.3; whole lines, 247 launches, 1.06 times as long plain;
// one column each / four: 17 codebooks, M = 2890 N = 8936 53.8 / 35.8, 96, 2091 N = 10864 65.1 / 51.3, 640, 1754 N = 9000 123 / 118.
bool streaming_stores(uint32_t n, uint32_t M, uint32_t cb16)
{
    return M % 4 == 0 && (M % 16 == 0 || (uint64_t)n * M * 4 < SP_BLOCK_OUTPUT || (uint64_t)cb16 * 16 * M > 4000000);
}

template <int TN, int TM, int GS, int NW, bool WIDE, int KS, bool BLOCKS>
int launch_sparse_as(Ctx* ctx, const Amm& a, const uint8_t* d_idx, float* d_out, int32_t* d_acc, uint32_t n,
                     const Epilogue& ep)
{
    constexpr int LDS = sp_lds_bytes(TN, TM, GS, NW, WIDE, KS);
    constexpr int PER_CU = sp_wgs_per_cu(TN, TM, GS, NW, WIDE);
    static_assert(PER_CU * LDS <= 160 * 1024, "the CU's LDS holds the workgroups that its registers hold");
    constexpr int TOK_ITEM = sp_tok_item(TM, NW / KS);
    using Map = std::conditional_t<BLOCKS, XcdBlocks, XcdMap>;
    auto kernel_for = [](auto map) {
        using K = void (*)(const uint8_t*, const int8_t*, float*, int32_t*, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, Epilogue, decltype(map));
        if constexpr (BLOCKS) return static_cast<K>(gather_sparse_blocks_kernel<TN, TM, GS, NW>);
        else return static_cast<K>(gather_sparse_kernel<TN, TM, GS, NW, WIDE, KS>);
    };
    const auto streamed = kernel_for(Map{});
    const auto plain = kernel_for(PlainStores<Map>{});
    const uint32_t cb16 = sparse_codebooks(a.g);  // codebooks of 16 centroids in the tiled table
    const bool stream = streaming_stores(n, a.g.M, cb16);
    if (int rc = allow_dynamic_lds(ctx, stream ? reinterpret_cast<const void*>(streamed) : reinterpret_cast<const void*>(plain), LDS, "hipFuncSetAttribute(gather_sparse)")) return rc;
    const uint32_t n_token_tiles = (n + TOK_ITEM - 1) / TOK_ITEM;
    const uint32_t n_items = n_token_tiles * (a.g.M_pad / (16 * TN));
    uint32_t grid = ctx->prop.multiProcessorCount * PER_CU;
    if (grid > n_items) grid = n_items;
    // Outputs of 16 MiB and more: an XCD takes its token tiles in blocks of about 1024 tokens (2048 with
    // 64-column tiles) through all of its columns, so that the rows it is writing are written whole within a short time,
    // instead of a few columns of all of its rows.  With more tokens to a block fewer workgroups share the rows, with fewer
    // every column's table is fetched again for each of them.  us a pass over three operators, inputs and outputs in turn (one output written
    // over and over stays in the last cache up to 256 MiB, and shows nothing of this), 64-column tiles, three workgroups per CU, without blocks
    // and with blocks of 512, 1024, 2048, 4096 tokens: 768 -> 3072 N = 4096 33.8 / 29.9 30.0 30.2 30.6, N = 8192 54.8 / 50.2 50.1 50.0 49.9, N = 16384
    // 99 / 95 95 95 95; 2048 -> 2048 N = 16384 167 / 153 154 156 159; 1024 -> 4096 N = 8192 80 / 76 77 78 76; 3072 -> 768 N = 16384 124 / 119 119 119 120.
    // Without a column split by XCD smaller blocks cost more (1024 -> 4096 N = 32768, split over 1 / 8: 323 / 298 with 512 tokens, 323 / 301 with 2048).
    // Below 16 MiB there is no difference (768 -> 768, N = 2048 .. 4096).
    const uint32_t col_tiles = a.g.M_pad / (16 * TN);
    const XcdMap dealt = choose_xcd_map(col_tiles, n_token_tiles, grid, (uint64_t)cb16 * 16 * a.g.M_pad,
                                        (uint64_t)n * a.g.idx_row_bytes, a.g.tune_xcd_col_split);
    const auto xmap = [&] {
        if constexpr (BLOCKS) return xcd_blocks(dealt, col_tiles, n_token_tiles, (TN == 4 ? 2048 : 1024) / TOK_ITEM);
        else return dealt;
    }();
    if (BLOCKS) snprintf(a.last_gather, sizeof(a.last_gather), "gather_sparse_blocks_kernel<%d, %d, %d, %d>", TN, TM, GS, NW);
    else if (KS == 1) snprintf(a.last_gather, sizeof(a.last_gather), "gather_sparse_kernel<%d, %d, %d, %d, %s>", TN, TM, GS, NW, WIDE ? "true" : "false");
    else snprintf(a.last_gather, sizeof(a.last_gather), "gather_sparse_kernel<%d, %d, %d, %d, %s, %d>", TN, TM, GS, NW, WIDE ? "true" : "false", KS);
    a.note_launch(GS, LDS, TOK_ITEM, NW * 64);
    auto launch = [&](auto kern, const auto& map) {
        hipLaunchKernelGGL(kern, dim3(grid), dim3(NW * 64), LDS, ctx->stream, d_idx, reinterpret_cast<const int8_t*>(a.d_lut),
                           d_out, d_acc, n, a.g.M, cb16, a.g.idx_row_bytes, n_token_tiles, n_items, ep, map);
    };
    if (stream) launch(streamed, xmap);
    else launch(plain, PlainStores<Map>{xmap});
    return hip_check(ctx, hipGetLastError(), "gather_sparse_kernel launch");
}

template <int TN, int TM, int GS, int NW = 4, bool WIDE = false, int KS = 1>
int launch_sparse_tm(Ctx* ctx, const Amm& a, const uint8_t* d_idx, float* d_out, int32_t* d_acc, uint32_t n, const Epilogue& ep)
{
    // (17..32 centroids are here on request only, and a split of the codebooks is for launches of one round)
    if constexpr (!WIDE && KS == 1)
        if ((uint64_t)n * a.g.M * 4 >= SP_BLOCK_OUTPUT) return launch_sparse_as<TN, TM, GS, NW, WIDE, KS, true>(ctx, a, d_idx, d_out, d_acc, n, ep);
    return launch_sparse_as<TN, TM, GS, NW, WIDE, KS, false>(ctx, a, d_idx, d_out, d_acc, n, ep);
}

// 256- or 128-token items, whichever gives the shorter launch (the rule of the dense kernel)
template <int TN, bool WIDE>
int launch_sparse_tn(Ctx* ctx, const Amm& a, const uint8_t* d_idx, float* d_out, int32_t* d_acc, uint32_t n, const Epilogue& ep)
{
    const uint32_t cb16 = sparse_codebooks(a.g);
    const uint64_t col_tiles = a.g.M_pad / (16 * TN);
    const uint64_t items4 = (uint64_t)((n + sp_tok_item(4) - 1) / sp_tok_item(4)) * col_tiles;
    const uint64_t items2 = (uint64_t)((n + sp_tok_item(2) - 1) / sp_tok_item(2)) * col_tiles;
    const uint64_t slots = 2ull * ctx->prop.multiProcessorCount;
    bool small_items = prefer_small_items(items4, items2, slots);
    if (a.g.tune_token_item) small_items = a.g.tune_token_item == 128;
    // 48-column tiles read the sparse operand of a token group for three column groups only, so the copies and
    // the per-slice costs weigh most there: with eight waves per workgroup a slice is copied once per 512 tokens
    // and can be 64 codebooks deep (measured 44.1 -> 42.4 us at 3072 -> 768, N = 8192; the 96-column kernel
    // loses 3 us the same way, its two waves of a SIMD then waiting at the same barrier).  Taken where it gives the
    // shorter launch: a round of 512-token items takes 0.96 of a round of twice as many 256-token items, but a partly
    // filled last round costs a whole one (its workgroups are alone on their CUs either way), where four-wave
    // workgroups speed up (grid_rounds): the fused Q/K/V gather at N = 4096 (1.5 rounds) takes 21.7 us with four
    // waves and 27.4 us with eight.
    if constexpr (TN == 3 && !WIDE) {
        const uint64_t cus = ctx->prop.multiProcessorCount;
        const uint64_t items8 = (uint64_t)((n + sp_tok_item(4, 8) - 1) / sp_tok_item(4, 8)) * col_tiles;
        // (sums of fewer than 384 codebooks that three workgroups per CU take: 768 -> 2304 N = 8192 49.7 us a pass with eight waves, 46.2 with
        // them, 768 -> 3072 59.3 / 55.9; 3072 -> 768 N = 16384 124.2 / 127.2)
        if (!a.g.tune_token_item && !a.g.tune_cb_per_slice && cb16 % 64 == 0 && !small_items && items8 >= cus &&
            !(cb16 < 384 && sparse_three_per_cu(items4, cb16, cus)) &&
            0.96 * (double)((items8 + cus - 1) / cus) < grid_rounds(items4, slots))
            return launch_sparse_tm<TN, 4, 64, 8>(ctx, a, d_idx, d_out, d_acc, n, ep);
        // A launch of long sums that offers about one 256-token item per CU: 128-token items would fill the chip's
        // workgroup slots but copy every slice twice as often and re-read every table entry for two token groups
        // instead of four; with the codebooks of a slice split between the two waves of a SIMD the 256-token item
        // keeps both (3072 -> 768: N = 4096 26.3 -> 23.1 us, N = 3072 24.6 -> 22.6; half a round of such items
        // (N = 2048) or more than one (N = 6144), and sums of 192 codebooks, are not faster that way).
        if ((a.g.tune_token_item == 256 && a.g.tune_cb_per_slice == 64 && cb16 % 64 == 0) ||
            (!a.g.tune_token_item && !a.g.tune_cb_per_slice && cb16 % 64 == 0 && cb16 >= 384 && items4 <= cus &&
             10 * items4 >= 7 * cus))
            return launch_sparse_tm<TN, 4, 64, 8, false, 2>(ctx, a, d_idx, d_out, d_acc, n, ep);
    }
    if constexpr (!WIDE) if (a.g.tune_token_item == 512) {  // one workgroup of eight waves per CU
        if constexpr (TN == 3) {
            if (cb16 % 64 == 0 && a.g.tune_cb_per_slice == 64) return launch_sparse_tm<TN, 4, 64, 8>(ctx, a, d_idx, d_out, d_acc, n, ep);
        }
        // (CB_pad is a multiple of 32; 48-column tiles have no 16-codebook variant here: 12 blocks for 8 waves)
        if (TN == 3 || a.g.tune_cb_per_slice != 16) return launch_sparse_tm<TN, 4, 32, 8>(ctx, a, d_idx, d_out, d_acc, n, ep);
        if constexpr (TN != 3) return launch_sparse_tm<TN, 4, 16, 8>(ctx, a, d_idx, d_out, d_acc, n, ep);
    }
    if constexpr (TN <= 4 && !WIDE)
        if (!a.g.tune_token_item && !a.g.tune_cb_per_slice && sparse_three_per_cu(items4, cb16, ctx->prop.multiProcessorCount))
            return launch_sparse_tm<TN, 4, 16>(ctx, a, d_idx, d_out, d_acc, n, ep);
    constexpr int GSB = TN <= 4 ? 32 : 16;  // 32-codebook slices in two buffers where two workgroups still fit a CU
    if constexpr (GSB != 16) {
        if (cb16 % GSB == 0 && a.g.tune_cb_per_slice != 16) {
            if (small_items) return launch_sparse_tm<TN, 2, GSB, 4, WIDE>(ctx, a, d_idx, d_out, d_acc, n, ep);
            return launch_sparse_tm<TN, 4, GSB, 4, WIDE>(ctx, a, d_idx, d_out, d_acc, n, ep);
        }
    }
    if (small_items) return launch_sparse_tm<TN, 2, 16, 4, WIDE>(ctx, a, d_idx, d_out, d_acc, n, ep);
    return launch_sparse_tm<TN, 4, 16, 4, WIDE>(ctx, a, d_idx, d_out, d_acc, n, ep);
}

}  // namespace

uint32_t sparse_lds_bytes(uint32_t tn, bool wide) { return (uint32_t)sp_lds_bytes((int)tn, 4, 16, 4, wide); }

int launch_gather_sparse(Ctx* ctx, const Amm& a, const uint8_t* d_idx, float* d_out, int32_t* d_acc, uint32_t n,
                         float scale, float lut_bias_term)
{
    Epilogue ep;
    ep.scale = scale;
    ep.lut_bias_term = lut_bias_term;
    ep.bias = a.d_bias;
    ep.act = a.desc.activation;
    ep.op_scales = a.d_op_scales;
    ep.op_col_tiles = a.op_col_tiles;
    ep.op_idx_stride = a.op_idx_stride;
    if (a.g.C_tile == 32) {
        switch (a.g.q) {
            case 3: return launch_sparse_tn<3, true>(ctx, a, d_idx, d_out, d_acc, n, ep);
            case 4: return launch_sparse_tn<4, true>(ctx, a, d_idx, d_out, d_acc, n, ep);
            case 6: return launch_sparse_tn<6, true>(ctx, a, d_idx, d_out, d_acc, n, ep);
        }
    } else {
        switch (a.g.q) {
            case 3: return launch_sparse_tn<3, false>(ctx, a, d_idx, d_out, d_acc, n, ep);
            case 4: return launch_sparse_tn<4, false>(ctx, a, d_idx, d_out, d_acc, n, ep);
            case 6: return launch_sparse_tn<6, false>(ctx, a, d_idx, d_out, d_acc, n, ep);
        }
    }
    return set_error(ctx, PIMDL_ERR_UNSUPPORTED, "no sparse gather kernel for %u column groups", a.g.q);
}

}  // namespace pimdl
