// Body of gather_sparse_kernel and gather_sparse_blocks_kernel (gather_sp_kernel.hip), included inside each of them and nowhere else.  It
// takes from the kernel: the template's TN, TM, GS, NW, WIDE and KS, the arguments idx, lut, out, acc_out, N, M, CB_pad, idx_row_bytes,
// n_token_tiles, n_items and ep, and xmap, whose type is all that the two differ in: decode(position, n_token_tiles, column tile, token
// tile), which is also called for the position behind a workgroup's last item and must return then, with any values.
    constexpr int SP_WAVES = NW;
    constexpr int NWT = NW / KS;                   // waves with tokens of their own
    static_assert(KS == 1 || (KS == 2 && NW == 8), "the codebook split is between the two waves of a SIMD");
    constexpr int TOK_ITEM = sp_tok_item(TM, NWT);
    static_assert(TM == 4 || TM == 2, "a wave owns a whole or half a 64-token index block");
    constexpr int WN = 16 * TN;                    // columns per item
    constexpr int G = GS;                          // codebooks per slice
    constexpr int SLICE = G * WN * 16;             // bytes of one codebook slice
    constexpr int KSTEPS = G / 8 / KS;             // one instruction covers 8 codebooks (this wave's share of a slice)
    constexpr int IWORDS = G / 8 / KS;             // 32-bit index words per token and slice (8 nibbles each), this wave's
    constexpr int IWORDS_ALL = G / 8;
    constexpr int NBLK = SLICE / 1024;             // 1 KB blocks (one copy instruction of a wave) per slice
    constexpr int DMA_PER_WAVE = (NBLK + SP_WAVES - 1) / SP_WAVES;
    static_assert(KSTEPS >= 2, "the operand pipeline below re-arms inside a slice");

    // LDS: value table(s) | position words (1 KB) | NBUF LUT slice buffers | NIBUF index buffers
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    constexpr int NBUF = sp_nbuf(TN, TM, GS, NW, WIDE), NIBUF = NBUF;
    constexpr int PD = NBUF - 1;  // prefetch distance of the LUT stream, in slices
    constexpr uint32_t POS0 = sp_value_table_bytes(WIDE);  // position words
    constexpr uint32_t BUF0 = sp_table_bytes(WIDE);
    constexpr uint32_t IBUF0 = BUF0 + NBUF * SLICE;
    constexpr uint32_t IBYTES = sp_ix_blocks(TM, NWT) * 64 * 4 * IWORDS_ALL;   // index bytes of one slice (64-token blocks)
    constexpr uint32_t IWAVE = 64 * 4 * IWORDS_ALL;           // ... of one 64-token block
    // index words: one operation copies one word of 64 tokens (64 lanes x 4 B) or, where a slice has a multiple of
    // four words, four of them (64 lanes x 16 B: consecutive words of a 64-token block are consecutive 256-byte
    // pieces in the tiled index buffer and in LDS alike); fewer instructions, the same time (measured)
    constexpr bool IX_WIDE = IWORDS % 4 == 0;
    constexpr int IX_OPS = IX_WIDE ? IWORDS / 4 : IWORDS;
    constexpr int DMA_OPS = DMA_PER_WAVE + IX_OPS;            // memory operations per wave and slice
    // Up to 16 centroids: the value bytes of a nibble are 1 << 16 (c / 4) as a 64-bit number, made by one shift
    // instead of read from a table (one LDS read per token group and K-step instead of three; measured 1 - 7 %
    // of the kernel, most on narrow column tiles).
    constexpr bool VALU_VALUES = !WIDE;
    constexpr int A_OPS = VALU_VALUES ? 1 : 3;                // LDS reads per token group for the sparse operand

    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t tw = KS == 1 ? wave : wave % NWT;  // which tokens of the item
    const uint32_t kh = KS == 1 ? 0u : wave / NWT;    // which part of a slice's codebooks
    const uint32_t j = lane & 15;  // token within a group (sparse operand) / column within a group (dense operand, result)
    const uint32_t g = lane >> 4;
    if (blockIdx.x >= n_items) return;  // whole workgroup
    const uint32_t nslices = CB_pad / G;
    const uint32_t my_items = (n_items - blockIdx.x + gridDim.x - 1) / gridDim.x;
    const uint32_t total = my_items * nslices;

    // Table entry c (16 bytes): value bytes of a codebook whose centroid is c (first slot of group c / 4 is 1).
    // Position table, word b: the position bits of both codebooks of index byte b (c % 4 at value slot 2 (c / 4),
    // two bits per slot; low nibble in the low half of the word, high nibble in the high half).
    // WIDE: table h (h = 0, 1; 512 bytes each) has entry c at byte b = 16 h + c and zero entries elsewhere.
    static_assert(NW * 64 >= 256, "one table word per thread");
    if (WIDE && threadIdx.x < 256) {
        const uint32_t b = (threadIdx.x >> 2) & 31, table = threadIdx.x >> 7;
        const uint32_t c = b & 15, w = threadIdx.x & 3, grp = c >> 2;
        uint32_t word;
        if (w < 2) word = (grp >> 1) == w ? (1u << (16 * (grp & 1))) : 0u;  // value bytes 0..3 / 4..7: slot 2 grp
        else word = 0;
        if (WIDE && (b >> 4) != table) word = 0;
        reinterpret_cast<uint32_t*>(smem)[threadIdx.x] = word;
    }
    if (threadIdx.x < 256) {
        const uint32_t b = threadIdx.x;
        auto pos_bits = [](uint32_t c) { return (c & 3u) << (4 * (c >> 2)); };
        // WIDE: the byte is one centroid of 32; its bits belong to the half its table is looked up for
        const uint32_t word = WIDE ? pos_bits(b & 15) << (16 * ((b >> 4) & 1)) : pos_bits(b & 15) | (pos_bits(b >> 4) << 16);
        reinterpret_cast<uint32_t*>(smem + POS0)[b] = word;
    }

    auto col_of = [&](uint32_t p) { uint32_t c, t; xmap.decode(p, n_token_tiles, c, t); return c; };
    auto tok_tile_of = [&](uint32_t p) { uint32_t c, t; xmap.decode(p, n_token_tiles, c, t); return t; };
    uint32_t lut_item = blockIdx.x, lut_s = 0, ix_item = blockIdx.x, ix_s = 0;
    const int8_t* dma_base;   // uniform: start of the slice at the LUT stream position
    const uint8_t* ix_base;   // uniform: the 256-byte block of index words at the index stream position
    uint32_t ix_lane_off;
    auto locate_lut = [&]() { dma_base = lut + (size_t)col_of(lut_item) * CB_pad * (WN * 16); };
    const uint32_t last_block = (N - 1) / 64;
    auto locate_ix = [&]() {
        uint32_t blk = (tok_tile_of(ix_item) * TOK_ITEM + tw * (TM * 16)) / 64;
        if (blk > last_block) blk = last_block;  // clamp: results of such tokens are never stored
        const uint32_t op = ep.op_col_tiles ? col_of(ix_item) / ep.op_col_tiles : 0u;
        ix_base = idx + (size_t)op * ep.op_idx_stride + (size_t)blk * idx_row_bytes * 64;
        ix_lane_off = lane * (IX_WIDE ? 16 : 4) + kh * (IWORDS * 256);  // this wave's words of the block
    };
    // A wave copies DMA_PER_WAVE consecutive 1 KB blocks of a slice.  All of a slice's operations share one
    // global address (the wave's part of the slice, per lane) and one LDS address; the block is chosen by the
    // instruction's immediate offset, which the hardware adds to both.  The offset field reaches 4 KB, so blocks
    // beyond the fourth go through a second address pair 4 KB further on.
    // fetch = false (past the end of the stream): the operations re-copy the first slice of the table into a
    // buffer nobody reads any more, so that every slice issues the same number of operations and the waits
    // can count them.
    static_assert(NBLK % SP_WAVES == 0 && DMA_PER_WAVE <= 8, "whole blocks per wave, two address pairs");
    const uint32_t dma_wave = wave * (DMA_PER_WAVE * 1024);
    const uint32_t dma_lane = dma_wave + lane * 16;
    const int8_t* lut_src = nullptr;  // this slice's source for this lane
    uint32_t lut_dst = 0;             // ... and the wave's destination in LDS
    // buf_off: byte offset of the destination buffer among the slice buffers
    auto lut_begin = [&](uint32_t buf_off, bool fetch) {
        // the choice is uniform: made once on the scalar side, not per lane
        const int8_t* base = uniform_ptr(fetch ? dma_base : lut);
        lut_src = base + dma_lane;
        lut_dst = BUF0 + buf_off + dma_wave;
    };
    auto lut_op = [&](auto uc) {
        constexpr int u = decltype(uc)::value, hi = u / 4, lo = u % 4;
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(lut_src + hi * 4096),
                                         (__attribute__((address_space(3))) void*)(smem + lut_dst + hi * 4096), 16, lo * 1024, 0);
    };
    auto lut_advance = [&]() {
        dma_base += SLICE;
        if (++lut_s == nslices) {
            lut_s = 0;
            lut_item += gridDim.x;
            locate_lut();  // may point past the last item; never dereferenced then
        }
    };
    auto stage_lut = [&](uint32_t buf) {
        lut_begin(buf * SLICE, true);
        static_for<0, DMA_PER_WAVE>([&](auto uc) { lut_op(uc); });
        lut_advance();
    };
    // index words: the same scheme, 256 bytes (64 tokens x one word) per operation
    const uint8_t* ix_src = nullptr;
    uint32_t ix_dst = 0;
    auto ix_begin = [&](uint32_t ibuf_off, bool fetch) {
        const uint8_t* base = uniform_ptr(fetch ? ix_base : idx);  // idx itself: any 64 tokens' words, never read
        ix_src = base + ix_lane_off;
        ix_dst = IBUF0 + ibuf_off + (tw * (TM * 16) / 64) * IWAVE + kh * (IWORDS * 256);
    };
    auto ix_op = [&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if constexpr (IX_WIDE)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)ix_src,
                                             (__attribute__((address_space(3))) void*)(smem + ix_dst), 16, 1024 * i, 0);
        else
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)ix_src,
                                             (__attribute__((address_space(3))) void*)(smem + ix_dst), 4, 256 * i, 0);
    };
    auto ix_advance = [&]() {
        ix_base += IWORDS_ALL * 256;
        if (++ix_s == nslices) {
            ix_s = 0;
            ix_item += gridDim.x;
            if (ix_item < n_items) locate_ix();
        }
    };
    auto stage_ix = [&](uint32_t ibuf) {
        ix_begin(ibuf * IBYTES, true);
        static_for<0, IX_OPS>([&](auto ic) { ix_op(ic); });
        ix_advance();
    };
    // Index word k of a token holds the nibbles of codebooks 8k .. 8k+7 of the slice; this lane's two are byte g,
    // which it reads on its own (the four lane groups read the four bytes of the same word: one bank, broadcast).
    // Kept as the two table offsets, nibble * 16.
    const uint32_t ix_lane = IBUF0 + (tw * (TM * 16) / 64) * IWAVE + kh * (IWORDS * 256) + (((tw * (TM * 16)) & 63) + j) * 4 + g;
    auto read_ix = [&](uint32_t (&raw)[TM][IWORDS], uint32_t ibuf_off) {
        const uint32_t addr = ix_lane + ibuf_off;
        static_for<0, TM * IWORDS>([&](auto ec) {
            constexpr int t = decltype(ec)::value / IWORDS, i = decltype(ec)::value % IWORDS;
            lds_read_u8<(i * 64 + t * 16) * 4>(raw[t][i], addr);
        });
    };
    // the index bytes requested by read_ix have landed (the registers pass through the wait)
    auto wait_ix = [&](uint32_t (&raw)[TM][IWORDS]) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int t = 0; t < TM; ++t)
#pragma unroll
            for (int i = 0; i < IWORDS; ++i) asm volatile("" : "+v"(raw[t][i]));
    };

    v4i acc[TM][TN];
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int c = 0; c < TN; ++c) acc[t][c] = (v4i){0, 0, 0, 0};

    // ---- epilogue ------------------------------------------------------------------------------------
    // Lane (g, j) holds acc[t][c][r] = sum for token 16 t + 4 g + r and the column that sparse_tile_column
    // assigns to position 16 c + j.  Pieces of W = 4, 2 or 1 groups give W consecutive columns per lane.
    constexpr int N4 = TN / 4 * 4, N2 = N4 + (TN % 4) / 2 * 2;
    constexpr int NPIECES = TN / 4 + (TN % 4) / 2 + TN % 2;
    constexpr int EPI_STORES = TM * 4 * NPIECES;  // stores of a wave in the epilogue of a full tile
    auto epilogue_as = [&](uint32_t item, auto actc) __attribute__((always_inline)) -> bool {
        constexpr bool ACT = decltype(actc)::value;
        uint32_t je = j, ge = g;
        asm volatile("" : "+v"(je), "+v"(ge));  // keeps the address arithmetic below out of the slice loop
        const uint32_t colblk = col_of(item);
        Epilogue epl = ep;
        if (ep.op_col_tiles) epl.scale = scalar_load1(ep.op_scales + colblk / ep.op_col_tiles);
        const uint32_t tile_tok0 = tok_tile_of(item) * TOK_ITEM;
        const uint32_t tok0 = tile_tok0 + tw * (TM * 16) + 4 * ge;
        const bool full = !acc_out && tile_tok0 + TOK_ITEM <= N && (colblk + 1) * WN <= M;
        auto piece = [&](auto c0c, auto wc) __attribute__((always_inline)) {
            constexpr int c0 = decltype(c0c)::value, W = decltype(wc)::value;
            const uint32_t f = colblk * WN + 16 * c0 + W * je;  // first of this lane's W columns
            float bv[W];
#pragma unroll
            for (int e = 0; e < W; ++e) bv[e] = (ep.bias && f + e < M) ? ep.bias[f + e] : 0.0f;
#pragma unroll
            for (int t = 0; t < TM; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t tok = tok0 + t * 16 + r;
                    float o[W];
                    int32_t a[W];
#pragma unroll
                    for (int e = 0; e < W; ++e) {
                        a[e] = acc[t][c0 + e][r];
                        o[e] = dequant<ACT>(a[e], epl, bv[e]);
                    }
                    float* dst = out + (size_t)tok * M + f;
                    if (full) {  // workgroup-uniform: every token and column of the tile exists
                        if constexpr (!STREAM) {  // (see streaming_stores)
                            typedef float vf __attribute__((ext_vector_type(W), aligned(4)));  // columns of a row of any width: dword alignment only
                            vf v;
#pragma unroll
                            for (int e = 0; e < W; ++e) v[e] = o[e];
                            *reinterpret_cast<vf*>(dst) = v;
                        } else if constexpr (W == 4) {
                            typedef float v4f __attribute__((ext_vector_type(4)));
                            // Streaming stores; 96-column tiles, which only a caller that names them takes, plain ones.  (Measured over
                            // one output written again and again, when 96 columns were the choice at 768 -> 3072: 0.7 us faster there, N =
                            // 8192, 100 MB, and 1.4 us slower in the 48 columns of 3072 -> 768, 25 MB.)
                            if constexpr (TN == 6) *reinterpret_cast<v4f*>(dst) = (v4f){o[0], o[1], o[2], o[3]};
                            else __builtin_nontemporal_store((v4f){o[0], o[1], o[2], o[3]}, reinterpret_cast<v4f*>(dst));
                        } else if constexpr (W == 2) {
                            typedef float v2f __attribute__((ext_vector_type(2)));
                            __builtin_nontemporal_store((v2f){o[0], o[1]}, reinterpret_cast<v2f*>(dst));
                        } else {
                            __builtin_nontemporal_store(o[0], dst);
                        }
                        continue;
                    }
                    if (tok >= N) continue;
#pragma unroll
                    for (int e = 0; e < W; ++e)
                        if (f + e < M) {
                            dst[e] = o[e];
                            if (acc_out) acc_out[(size_t)tok * M + f + e] = a[e];
                        }
                }
        };
        static_for<0, TN / 4>([&](auto pc) { piece(std::integral_constant<int, 4 * decltype(pc)::value>{}, std::integral_constant<int, 4>{}); });
        if constexpr (N2 > N4) piece(std::integral_constant<int, N4>{}, std::integral_constant<int, 2>{});
        if constexpr (TN > N2) piece(std::integral_constant<int, N2>{}, std::integral_constant<int, 1>{});
#pragma unroll
        for (int t = 0; t < TM; ++t)
#pragma unroll
            for (int c = 0; c < TN; ++c) acc[t][c] = (v4i){0, 0, 0, 0};
        return full;
    };
    auto epilogue = [&](uint32_t item) __attribute__((always_inline)) -> bool {
        return ep.act == PIMDL_ACT_GELU_TANH ? epilogue_as(item, std::true_type{}) : epilogue_as(item, std::false_type{});
    };

    // ---- prologue: slices 0 .. PD-1, index words 0 .. PD ------------------------------------------------
    locate_lut();
    locate_ix();
    static_for<0, PD + 1>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if (i < total) stage_ix(i);
    });
    static_for<0, PD>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if (i < total) stage_lut(i);
    });
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();  // also: the table is complete
    uint32_t iw_raw[TM][IWORDS];
    read_ix(iw_raw, 0);
    wait_ix(iw_raw);

    uint32_t item0 = blockIdx.x;
    // this lane's 16 bytes of codebook g (of this wave's share of the slice), column position j
    const uint32_t b_lane = BUF0 + (g * WN + j) * 16 + kh * (KSTEPS * 8 * WN * 16);
    // byte offsets of the buffers in their rings: the slice being read and the one its copies go into (the
    // slice before), the index words read next and the ones copied into
    uint32_t cur_off = 0, copy_off = (NBUF - 1) * SLICE, ixn_off = IBYTES, ixc_off = 0;
    uint32_t k = 0;
    bool stores_behind = false;
    constexpr bool COUNT_STORES = (PD - 1) * DMA_OPS + EPI_STORES <= 63;  // memory counter range

    for (uint32_t it = 0; it < my_items; ++it, item0 += gridDim.x) {
    for (uint32_t s0 = 0; s0 < nslices; ++s0, ++k) {
        // at most the operations issued during the previous PD-1 slices are outstanding: this wave's share of
        // slice k (and of index words k+1) has landed; after the barrier everybody's has, and everybody is
        // done with slice k-1, whose buffer slice k+PD goes into
        if (k != 0) {
            if (COUNT_STORES && stores_behind) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(COUNT_STORES ? (PD - 1) * DMA_OPS + EPI_STORES : 0) : "memory");
            else asm volatile("s_waitcnt vmcnt(%0)" ::"n"((PD - 1) * DMA_OPS) : "memory");
            stores_behind = false;
            __syncthreads();
        }
        const bool fetch = k + PD < total;
        const bool fetch_ix = k + PD + 1 < total;
        const uint32_t bbase = cur_off + b_lane;
        lut_begin(copy_off, fetch);
        ix_begin(ixc_off, fetch_ix);

        // Operand registers: the dense operand of a column group is re-armed with the next K-step's bytes as
        // soon as its TM instructions have been issued; the sparse operand is double buffered.
        v4i b_lo[TN], b_hi[TN];
        v2i a_lo[2][TM], a_hi[2][TM];
        int pw[2][TM];  // the lane's position word
        auto issue_b = [&](auto ksc, auto cc) {
            constexpr int ks = decltype(ksc)::value, c = decltype(cc)::value;
            lds_read<((8 * ks) * WN + c * 16) * 16>(b_lo[c], bbase);
            lds_read<((8 * ks + 4) * WN + c * 16) * 16>(b_hi[c], bbase);
        };
        // The sparse operand of K-step ks from the index bytes: what a byte turns into is worked out here, between the
        // matrix instructions of the K-step before (a few vector operations per token group in their shadow), not for
        // the whole slice at its boundary, where a wave would spend them alone.
        auto issue_a = [&](auto ksc) {
            constexpr int ks = decltype(ksc)::value;
#pragma unroll
            for (int t = 0; t < TM; ++t) {
                const uint32_t raw = iw_raw[t][ks];
                const uint32_t pa = raw << 2;  // its position word
                if constexpr (VALU_VALUES) {
                    // the shift that makes the value bytes: 16 bits per group of four centroids
                    const uint64_t v0 = 1ull << (pa & 0x30u), v1 = 1ull << ((raw >> 2) & 0x30u);
                    a_lo[ks & 1][t] = (v2i){(int)(uint32_t)v0, (int)(uint32_t)(v0 >> 32)};
                    a_hi[ks & 1][t] = (v2i){(int)(uint32_t)v1, (int)(uint32_t)(v1 >> 32)};
                } else {
                    // (17..32 centroids) the byte is one codebook's centroid: its entry in the first and in the second table
                    const uint32_t e0 = raw << 4;
                    lds_read64<0>(a_lo[ks & 1][t], e0);
                    lds_read64<512>(a_hi[ks & 1][t], e0);
                }
                lds_read32<POS0>(pw[ks & 1][t], pa);
            }
        };
        // slice prologue: sparse operand first, then the dense operand of every column group, in this order
        issue_a(std::integral_constant<int, 0>{});
        static_for<0, TN>([&](auto cc) { issue_b(std::integral_constant<int, 0>{}, cc); });

        static_for<0, KSTEPS>([&](auto ksc) {
            constexpr int ks = decltype(ksc)::value;
            constexpr bool LAST = ks + 1 == KSTEPS;
            constexpr int RI = TM * IWORDS;  // index-word reads issued after column group 0 of the last K-step
            static_for<0, TN>([&](auto cc) {
                constexpr int c = decltype(cc)::value;
                // LDS operations complete in order; the count is the number of operations issued after the
                // ones this column group needs (see the issue order above and below)
                if constexpr (c == 0) lgkm_wait<2 * (TN - 1)>();
                else if constexpr (LAST) lgkm_wait<2 * (TN - 1 - c) + RI>();
                else lgkm_wait<2 * TN + A_OPS * TM - 2>();
                if constexpr (c == 0) {
#pragma unroll
                    for (int t = 0; t < TM; ++t)
                        asm volatile("" : "+v"(a_lo[ks & 1][t]), "+v"(a_hi[ks & 1][t]), "+v"(pw[ks & 1][t]));
                }
                asm volatile("" : "+v"(b_lo[c]), "+v"(b_hi[c]));
                __builtin_amdgcn_sched_barrier(0);
                const v8i bb = {b_lo[c][0], b_lo[c][1], b_lo[c][2], b_lo[c][3], b_hi[c][0], b_hi[c][1], b_hi[c][2], b_hi[c][3]};
#pragma unroll
                for (int t = 0; t < TM; ++t) {
                    const v4i aa = {a_lo[ks & 1][t][0], a_lo[ks & 1][t][1], a_hi[ks & 1][t][0], a_hi[ks & 1][t][1]};
                    acc[t][c] = __builtin_amdgcn_smfmac_i32_16x16x128_i8(aa, bb, acc[t][c], pw[ks & 1][t], 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (!LAST) {
                    issue_b(std::integral_constant<int, ks + 1>{}, cc);
                    if constexpr (c == 0) issue_a(std::integral_constant<int, ks + 1>{});
                } else if constexpr (c == 0) {
                    read_ix(iw_raw, ixn_off);  // the next slice's index words (this wave's own copy, landed)
                }
                // this slice's copy operations (slice k+PD of the table, index words k+PD+1), a few per column group
                constexpr int IK = PD == 1 ? KSTEPS * TN / 2 : KSTEPS * TN;
                constexpr int pos = ks * TN + c;
                static_for<(pos < IK ? pos : IK) * DMA_OPS / IK, (pos + 1 < IK ? pos + 1 : IK) * DMA_OPS / IK>([&](auto oc) {
                    constexpr int o = decltype(oc)::value;
                    if constexpr (o < DMA_PER_WAVE) lut_op(std::integral_constant<int, o>{});
                    else ix_op(std::integral_constant<int, o - DMA_PER_WAVE>{});
                });
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        if (fetch) {
            lut_advance();
            if (fetch_ix) ix_advance();
        }
        wait_ix(iw_raw);

        copy_off = cur_off;
        cur_off = cur_off + SLICE == NBUF * SLICE ? 0 : cur_off + SLICE;
        ixc_off = ixn_off;
        ixn_off = ixn_off + IBYTES == NIBUF * IBYTES ? 0 : ixn_off + IBYTES;
    }
    if constexpr (KS == 2) {
        // the two halves of every sum meet in the slice buffer read last (nothing is copied into it before the next
        // slice's barrier): waves 4..7 put their accumulators there, waves 0..3 add them to their own
        static_assert(NWT * 64 * TM * TN * 16 <= SLICE, "the accumulators of half the waves fit a slice buffer");
        v4i* cbuf = reinterpret_cast<v4i*>(smem + BUF0 + copy_off) + tw * (TM * TN * 64) + lane;
        __syncthreads();  // every wave is done reading that buffer
        if (kh == 1) {
#pragma unroll
            for (int t = 0; t < TM; ++t)
#pragma unroll
                for (int c = 0; c < TN; ++c) {
                    cbuf[(t * TN + c) * 64] = acc[t][c];
                    acc[t][c] = (v4i){0, 0, 0, 0};
                }
        }
        __syncthreads();
        if (kh == 0) {
#pragma unroll
            for (int t = 0; t < TM; ++t)
#pragma unroll
                for (int c = 0; c < TN; ++c) acc[t][c] += cbuf[(t * TN + c) * 64];
            stores_behind = epilogue(item0);
        }
    } else {
        stores_behind = epilogue(item0);
    }
    }
