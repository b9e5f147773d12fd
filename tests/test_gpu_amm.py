"""Parity of the HIP path (through the C ABI) against the CPU oracle, on the same seeded inputs.

Bar: bit-exact centroid indices, bit-exact int32 accumulators, bit-exact fp32 output for the int8
path (the epilogue is three separately rounded fp32 operations on both sides); fp32-LUT path within
1e-5 relative (in fact also bit-exact, since both sides add in ascending codebook order)."""
import os

import numpy as np
import pytest

import oracle
from conftest import kernel_switches
from __graft_entry__ import load_package

pimdl = load_package()
pytestmark = pytest.mark.gpu

THREADS = 8


@pytest.fixture(scope="module")
def ctx():
    c = pimdl.Context(0)
    yield c
    c.close()


def make_case(seed, N, K, v, C, M, lut="i8", dist="normal"):
    rng = np.random.default_rng(seed)
    CB = K // v
    if dist == "normal":
        x = rng.standard_normal((N, K)).astype(np.float32)
        cent = rng.standard_normal((CB, C, v)).astype(np.float32)
    else:  # the reference driver's ranges (test_amm.cpp:26-45)
        x = rng.uniform(-5, 5, (N, K)).astype(np.float32)
        cent = rng.uniform(-10, 10, (CB, C, v)).astype(np.float32)
    bias = rng.standard_normal(M).astype(np.float32)
    if lut == "i8":
        table = rng.integers(-128, 128, (CB, C, M)).astype(np.int8)
    else:
        table = rng.standard_normal((CB, C, M)).astype(np.float32)
    return x, cent, table, bias


def check_i8(ctx, seed, N, K, v, C, M, scale=0.0123, lut_bias=0.0, bias_mode=0, dist="normal", max_n=None):
    x, cent, lut, bias = make_case(seed, N, K, v, C, M, "i8", dist)
    CB = K // v
    amm = ctx.amm(cent, lut, np.float32(scale), bias, max_n=max_n or N, lut_bias=lut_bias, bias_mode=bias_mode)
    out, idx, acc = amm.run_debug(x)
    want_idx = oracle.index_calculation(x, cent, v, threads=THREADS)
    want_acc = oracle.gather_i8(want_idx, lut, threads=THREADS)
    want_out = oracle.dequant(want_acc, bias, CB, scale, lut_bias, bias_mode, threads=THREADS)
    assert np.array_equal(idx, want_idx), f"indices: {(idx != want_idx).sum()} of {idx.size} differ"
    assert np.array_equal(acc, want_acc), f"accumulators: {(acc != want_acc).sum()} of {acc.size} differ"
    assert np.array_equal(out.view(np.uint32), want_out.view(np.uint32)), "fp32 output bits differ"
    # the plain entry point gives the same bytes as the debug one
    assert np.array_equal(amm.run(x).view(np.uint32), out.view(np.uint32))
    amm.close()


def test_config1_single_amm(ctx):
    """N=128, K=768, v=2 (384 codebooks), 16 centroids, M=768, LUT = quantised centroid x W."""
    rng = np.random.default_rng(0)
    N, K, v, C, M = 128, 768, 2, 16, 768
    CB = K // v
    x = rng.standard_normal((N, K)).astype(np.float32)
    cent = rng.standard_normal((CB, C, v)).astype(np.float32)
    W = (rng.standard_normal((K, M)) * 0.02).astype(np.float32)
    lut, scales = oracle.lut_quant(oracle.lutgen_f32(cent, W, threads=THREADS))
    bias = np.zeros(M, np.float32)
    want_out, want_idx, want_acc = oracle.amm_cpu(x, cent, lut, bias, v, float(scales[0]), 0.0, threads=THREADS)
    amm = ctx.amm(cent, lut, scales, bias, max_n=N)
    out, idx, acc = amm.run_debug(x)
    assert np.array_equal(idx, want_idx)
    assert np.array_equal(acc, want_acc)
    assert np.array_equal(out.view(np.uint32), want_out.view(np.uint32))
    amm.close()


@pytest.mark.parametrize("v,C", [(2, 8), (2, 16), (2, 32), (4, 8), (4, 16), (4, 32), (8, 8), (8, 16), (8, 32),
                                 (16, 16), (32, 16), (4, 64), (4, 128), (2, 256)])
def test_sweep_sub_vector_length_and_centroids(ctx, v, C):
    check_i8(ctx, 100 + v * 7 + C, N=300, K=64 * v if v < 16 else 96 * v // 2, v=v, C=C, M=200)


@pytest.mark.parametrize("N,K,v,C,M", [
    (1, 8, 4, 16, 4),        # smallest sensible shape
    (17, 24, 4, 16, 20),     # CB=6 (padded to 32), M not a multiple of the column block
    (255, 36, 4, 16, 63),    # M % 4 != 0: scalar stores
    (257, 40, 4, 5, 130),    # C not a power of two
    (513, 12, 3, 7, 33),     # sub_vec_len with no specialised kernel
    (64, 10, 5, 20, 18),     # generic v, 8-bit indices, K % 4 != 0
    (100, 6, 2, 16, 64),     # CB=3 (odd), K % 4 != 0: scalar activation loads
    (300, 44, 4, 20, 40),    # 17..32 centroids on the matrix-core search: ids past C never win
    (129, 18, 2, 17, 24),    # same, v=2, CB=9
    (200, 72, 8, 31, 50),    # same, v=8
    (333, 70, 10, 16, 52),   # sub_vec_len 10 (the reference's token_dim 2560 over 256 codebooks): CB=7, K % 4 != 0
    (130, 170, 10, 12, 37),  # ... CB=17 (two codebook tiles, the second ragged), C not a power of two
    (65, 640, 10, 40, 24),   # ... 8-bit indices, several centroid groups per codebook
    (257, 60, 20, 16, 20),   # sub_vec_len 20 (token_dim 5120): CB=3
    (100, 500, 20, 130, 16), # ... CB=25, more than 128 centroids
])
def test_ragged_shapes(ctx, N, K, v, C, M):
    check_i8(ctx, N + K + M, N, K, v, C, M)


@pytest.mark.parametrize("N,M", [
    (512, 768),     # 8 column tiles x 4 token tiles: one column tile per XCD
    (1000, 380),    # 4 column tiles x 8 token tiles (last one ragged): columns over 4, tokens over 2
    (2048, 192),    # 2 column tiles x 16 token tiles: columns over 2, tokens over 4
    (4096, 96),     # 1 column tile x 32 token tiles: tokens over 8
    (768, 768),     # 6 token tiles: no split divides, plain order
])
def test_every_item_is_computed_once_however_items_are_dealt_to_the_xcds(ctx, N, M):
    """The one-hot gather deals (column tile, token tile) items to the 8 XCDs by a split chosen per shape;
    a dropped or doubled item shows as wrong accumulators."""
    if os.environ.get("PIMDL_GATHER_ROWS") == "1":
        pytest.skip("the matrix-core gather is switched off")
    x, cent, lut, bias = make_case(N + M, N, 128, 4, 16, M)
    # (naming the items also keeps the kernel for few tokens away, which deals nothing to the XCDs)
    amm = ctx.amm(cent, lut, np.float32(0.01), bias, max_n=N, tuning={"col_block": 96, "token_item": 128})
    out, idx, acc = amm.run_debug(x)
    assert amm.last_gather_kernel().startswith(("gather_sparse_kernel<", "gather_onehot_kernel<")), amm.last_gather_kernel()
    assert amm.geometry()["tokens_per_wg"] == 128
    want_idx = oracle.index_calculation(x, cent, 4, threads=THREADS)
    want_acc = oracle.gather_i8(want_idx, lut, threads=THREADS)
    assert np.array_equal(idx, want_idx)
    assert np.array_equal(acc, want_acc)
    assert np.array_equal(out.view(np.uint32),
                          oracle.dequant(want_acc, bias, 32, 0.01, 0.0, 0, threads=THREADS).view(np.uint32))
    amm.close()


@pytest.mark.parametrize("C,lut,group", [(16, "i8", 0), (32, "i8", 0), (16, "f32", 0), (16, "i8", 4)])
def test_gelu_in_the_epilogue(ctx, C, lut, group):
    """activation=ACT_GELU_TANH: same indices and accumulators, output = tanh-GELU of the plain output
    (each of the gather kernels: matrix-core one-hot, byte adder, fp32 table, grouped scales)."""
    N, K, v, M = 300, 128, 4, 200
    x, cent, table, bias = make_case(C + group, N, K, v, C, M, lut)
    CB = K // v
    scales = None if lut == "f32" else (np.full((CB + group - 1) // group, 0.02, np.float32) if group else np.float32(0.02))
    plain = ctx.amm(cent, table, scales, bias, max_n=N, scale_group=group)
    fused = ctx.amm(cent, table, scales, bias, max_n=N, scale_group=group, activation=pimdl.ACT_GELU_TANH)
    y = plain.run(x).astype(np.float64)
    want = 0.5 * y * (1 + np.tanh(np.sqrt(2 / np.pi) * (y + 0.044715 * y ** 3)))
    got = fused.run(x)
    assert (np.abs(y) > 3).any() and (np.abs(y) < 0.1).any()  # both tails and the middle are exercised
    np.testing.assert_allclose(got, want, rtol=2e-6, atol=1e-7)
    if lut == "i8" and not group:
        _, idx, acc = fused.run_debug(x)
        _, idx0, acc0 = plain.run_debug(x)
        assert np.array_equal(idx, idx0) and np.array_equal(acc, acc0)
    # extreme inputs: -0 for very negative values (never NaN), identity for very positive ones
    big = ctx.amm(cent, table, scales, np.where(np.arange(M) % 2 == 0, 1e6, -1e6).astype(np.float32), max_n=N,
                  scale_group=group, activation=pimdl.ACT_GELU_TANH)
    raw = ctx.amm(cent, table, scales, np.where(np.arange(M) % 2 == 0, 1e6, -1e6).astype(np.float32), max_n=N,
                  scale_group=group)
    yb, y0 = big.run(x), raw.run(x)
    assert np.array_equal(yb[:, 0::2], y0[:, 0::2]) and not yb[:, 1::2].any() and not np.isnan(yb).any()
    for a in (plain, fused, big, raw):
        a.close()
    with pytest.raises(pimdl.PimdlError):
        ctx.amm(cent, table, scales, bias, max_n=N, scale_group=group, activation=7)


def test_reference_driver_value_ranges_and_bias_modes(ctx):
    # uniform(-5,5) activations, uniform(-10,10) centroids, scale 0.1, bias 0.2 as in the shipped YAML
    check_i8(ctx, 7, 256, 128, 4, 16, 96, scale=0.1, lut_bias=0.2, bias_mode=0, dist="uniform")
    check_i8(ctx, 8, 256, 128, 4, 16, 96, scale=0.1, lut_bias=0.2, bias_mode=1, dist="uniform")


def test_golden_reference_vectors_on_gpu(ctx, golden_index):
    """The fixtures produced by the reference's own compiled index_calculation."""
    for i in range(int(golden_index["ncases"])):
        x, cent, want = golden_index[f"c{i}_x"], golden_index[f"c{i}_cent"], golden_index[f"c{i}_idx"]
        CB, C, v = cent.shape
        lut = np.zeros((CB, C, 4), np.int8)
        amm = ctx.amm(cent, lut, np.float32(1.0), None, max_n=x.shape[0])
        got = amm.index_calculation(x)
        assert np.array_equal(got, want), f"golden case {i} ({golden_index[f'c{i}_kind']})"
        for key in golden_index.files:
            if key.startswith(f"c{i}_tiled_"):
                _, _, ns, cm = key.split("_")
                assert np.array_equal(amm.index_calculation(x, int(ns), int(cm)), golden_index[key]), key
        amm.close()


def test_near_ties_follow_the_scan_not_the_true_argmin(ctx):
    """Inputs midway between two centroids: many distance pairs differ by ~1e-6."""
    rng = np.random.default_rng(5)
    N, CB, C, v = 2048, 32, 16, 4
    cent = rng.standard_normal((CB, C, v)).astype(np.float32)
    a = rng.integers(0, C, (N, CB))
    b = (a + 1 + rng.integers(0, C - 1, (N, CB))) % C
    cb = np.arange(CB)[None, :]
    mid = (cent[cb, a] + cent[cb, b]) * np.float32(0.5)
    x = (mid + rng.standard_normal((N, CB, v)).astype(np.float32) * np.float32(2e-7)).reshape(N, CB * v)
    want = oracle.index_calculation(x, cent, v, threads=THREADS)
    true_argmin = oracle.np_distances(x, cent).argmin(-1)
    assert (want != true_argmin).sum() > 100  # the case really separates the two rules
    amm = ctx.amm(cent, np.zeros((CB, C, 4), np.int8), np.float32(1.0), None, max_n=N)
    assert np.array_equal(amm.index_calculation(x), want)
    amm.close()


@pytest.mark.parametrize("C", [16, 8, 5, 32, 20, 64])
def test_gather_from_given_indices_and_invariants(ctx, C):
    """C <= 8 runs the paired form of the matrix-core gather (two codebooks per index byte, odd CB), 17..32 the
    sparse form with every codebook as two of 16 (byte indices), more than 32 the byte adder."""
    rng = np.random.default_rng(21)
    N, CB, M, v = 300, 41 if C < 16 else 40, 192, 4
    cent = rng.standard_normal((CB, C, v)).astype(np.float32)
    lut = rng.integers(-128, 128, (CB, C, M)).astype(np.int8)
    idx = rng.integers(0, C, (N, CB)).astype(np.uint16)
    amm = ctx.amm(cent, lut, np.float32(1.0), None, max_n=N)
    out = amm.lut_gather(idx)
    want = oracle.gather_i8(idx, lut, threads=THREADS)
    assert np.array_equal(out, want.astype(np.float32))
    amm.close()
    # extremes: every entry -128 / +127, CB = 768 (the largest of the BERT shapes)
    CB = 768
    cent = rng.standard_normal((CB, C, v)).astype(np.float32)
    idx = rng.integers(0, C, (64, CB)).astype(np.uint16)
    for val in (-128, 127):
        amm = ctx.amm(cent, np.full((CB, C, 64), val, np.int8), np.float32(1.0), None, max_n=64)
        assert (amm.lut_gather(idx) == float(val * CB)).all()
        amm.close()


@pytest.mark.parametrize("C,v", [(16, 4), (8, 2), (32, 8)])
def test_fp32_lut_path(ctx, C, v):
    N, K, M = 300, 48 * v, 100
    x, cent, lut, bias = make_case(31 + C, N, K, v, C, M, "f32")
    amm = ctx.amm(cent, lut, None, bias, max_n=N)
    out, idx, _ = amm.run_debug(x)
    want_idx = oracle.index_calculation(x, cent, v, threads=THREADS)
    assert np.array_equal(idx, want_idx)
    want = oracle.gather_f32(want_idx, lut, bias, threads=THREADS)
    np.testing.assert_allclose(out, want, rtol=1e-5, atol=1e-6)  # the stated tolerance for fp32 paths
    amm.close()


@pytest.mark.parametrize("group,C,v,CB,M", [(1, 16, 4, 48, 100), (3, 16, 4, 48, 100), (5, 16, 2, 48, 64),
                                            (16, 16, 4, 192, 96), (64, 8, 8, 48, 33), (7, 32, 4, 40, 100),
                                            (4, 64, 4, 20, 72), (2, 256, 2, 6, 40)])
def test_scale_per_codebook_group(ctx, group, C, v, CB, M):
    """int8 LUT with one scale per `group` codebooks (an extension the reference does not have, so the
    only pin is the oracle's definition: int32 inside a group, then fp32 `tot += (float)acc_g * scale[g]`
    over groups ascending, then + bias).  Bit-exact against it, including ragged last groups, a group
    larger than CB, 4- and 8-bit index rows; group 1 is one scale per codebook."""
    N, K = 300, CB * v
    x, cent, lut, bias = make_case(500 + group + C, N, K, v, C, M)
    ng = (CB + group - 1) // group
    scales = np.random.default_rng(group).uniform(1e-3, 0.1, ng).astype(np.float32)
    amm = ctx.amm(cent, lut, scales, bias, max_n=N, scale_group=group)
    out = amm.run(x)
    want_idx = oracle.index_calculation(x, cent, v, threads=THREADS)
    want = oracle.gather_i8_grouped(want_idx, lut, scales, bias, group, threads=THREADS)
    assert np.array_equal(out.view(np.uint32), want.view(np.uint32)), \
        f"{(out.view(np.uint32) != want.view(np.uint32)).sum()} of {out.size} outputs differ"
    amm.close()


@pytest.mark.parametrize("C,M", [(64, 2752), (16, 2752), (130, 1376), (100, 1376), (40, 2750)])
@pytest.mark.parametrize("kind", ["f32", "grouped", "prescaled"])
def test_two_tokens_per_lane_in_the_fp32_table_gather(ctx, kind, C, M):
    """Wide outputs make the fp32-table gather of more than 32 centroids give each lane two tokens (rows t and t + 256 of a
    512-token block); the last block is ragged in both halves' sense: 1100 = 2 * 512 + 76.  (Up to 32 centroids the same sizes run on
    the kernel that reads its rows in pieces.)"""
    N, v, CB = 1100, 4, 8
    x, cent, lut, bias = make_case(77, N, CB * v, v, C, M, "f32" if kind == "f32" else "i8")
    want_idx = oracle.index_calculation(x, cent, v, threads=THREADS)
    if kind == "f32":
        amm = ctx.amm(cent, lut, None, bias, max_n=N)
        want = oracle.gather_f32(want_idx, lut, bias, threads=THREADS)
    else:
        group = 3 if kind == "grouped" else 1
        scales = np.random.default_rng(3).uniform(1e-3, 0.1, (CB + group - 1) // group).astype(np.float32)
        amm = ctx.amm(cent, lut, scales, bias, max_n=N, scale_group=group)
        want = oracle.gather_i8_grouped(want_idx, lut, scales, bias, group, threads=THREADS)
    assert np.array_equal(amm.run_debug(x, want_acc=False)[0].view(np.uint32), want.view(np.uint32))
    name = amm.last_gather_kernel()
    assert name.startswith("gather_f32_kernel<") and name.endswith(", 2>") if C > 32 else name.startswith("gather_f32_rows_kernel<"), name
    amm.close()


@pytest.mark.parametrize("N,K,v,C,Ms,lut", [
    (300, 256, 4, 16, (96, 200, 64), "i8"),     # tiled index rows (matrix-core gather), three outputs of different widths
    (1000, 128, 4, 8, (128, 128), "i8"),        # paired gather
    (1300, 128, 4, 8, (192, 192, 192), "i8"),   # paired gather, three members in one gather launch
    (700, 256, 4, 16, (96, 96), "i8"),          # one gather launch, 96-column tiles
    (2100, 128, 4, 16, (768, 768, 768), "i8"),  # the Q/K/V shape
    (257, 256, 2, 32, (100, 60), "i8"),         # 32 centroids: byte indices, tiled index rows (sparse gather, two tables)
    (900, 256, 4, 32, (96, 96, 96), "i8"),      # 32 centroids, three members in one gather launch
    (300, 256, 8, 16, (48, 80, 48), "f32"),     # fp32 tables
    (8192, 768, 4, 8, (768, 3072), "i8"),       # 8 centroids at a size where the wide member takes the sparse kernel, the narrow one the paired
    (8192, 256, 8, 8, (1536, 1536), "i8"),      # 8 centroids, both members on the sparse kernel, one gather launch
])
def test_operators_sharing_an_input_are_searched_by_one_launch(ctx, N, K, v, C, Ms, lut):
    """AmmGroup (separate Q/K/V projections): every output bit for bit that of the operator run alone."""
    if kernel_switches():
        pytest.skip("a kernel this test is about is switched off by the environment")
    rng = np.random.default_rng(N + K)
    x = rng.standard_normal((N, K)).astype(np.float32)
    amms = []
    for i, M in enumerate(Ms):
        _, cent, table, bias = make_case(900 + i, 1, K, v, C, M, lut)
        amms.append(ctx.amm(cent, table, None if lut == "f32" else np.float32(0.01 * (i + 1)), bias, max_n=N))
    group = ctx.amm_group(amms)
    outs = group.run(x)
    for a, o in zip(amms, outs):
        assert np.array_equal(o.view(np.uint32), a.run(x).view(np.uint32))
    if C == 8 and N == 8192:  # which kernel each member's launch rule took
        want_kernels = {(768, 3072): ("gather_onehot", "gather_sparse"), (1536, 1536): ("gather_sparse", "gather_sparse")}[Ms]
        for a, k in zip(amms, want_kernels):
            assert a.last_gather_kernel().startswith(k), (a.last_gather_kernel(), k)
    outs2 = group.run(x[:77])  # a smaller batch through the same group
    for o, o2 in zip(outs, outs2):
        assert np.array_equal(o[:77], o2)
    # one gather launch for all members where they are matrix-core gathers of one shape
    same_shape = lut == "i8" and C <= 32 and len(set(Ms)) == 1 and Ms[0] % amms[0].geometry()["col_block"] == 0
    assert (group.fused_cols > 0) == same_shape
    if same_shape:
        fused = group.run_fused(x)
        assert np.array_equal(fused.view(np.uint32), np.concatenate(outs, axis=1).view(np.uint32))
    else:
        with pytest.raises(pimdl.PimdlError):
            group.run_fused(x)
    group.close()
    for a in amms:
        a.close()


@pytest.mark.parametrize("CB,v,C,M,max_n,named", [
    (128, 2, 16, 1280, (9856, 9856, 9856), None),       # alone each takes 48 columns, which do not divide its width
    (128, 2, 16, 1216, (10400, 10400), None),
    (128, 2, 16, 1024, (1024, 1024, 1024), None), (32, 4, 12, 1024, (4608, 4608), None),
    (128, 2, 16, 768, (11008, 12608), None),            # 48 columns and 64
    (128, 2, 8, 1280, (9856, 10048, 4096), None),       # up to 8 centroids: tables of both one-hot kernels, two column tiles
    (128, 2, 16, 1280, (9856, 9856), {"col_block": 48}),   # a tile that the caller has named stays
    (128, 2, 16, 1280, (9856, 9856), {"token_item": 128}), (128, 2, 16, 1280, (9856, 9856), {"token_item": 256, "cb_per_slice": 64}),
    (32, 2, 16, 1000, (700, 700), None),                # no tile divides the width
])
def test_operators_side_by_side_take_a_column_tile_of_their_own(ctx, CB, v, C, M, max_n, named):
    """Whether operators share one gather launch depends on their width, not on the column tile that suits each of them alone at its
    largest batch: every column bit for bit that of the operator alone, at few tokens and many."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about the library's choice")
    import torch
    amms = []
    for i, n in enumerate(max_n):
        _, cent, lut, bias = make_case(5600 + i, 1, CB * v, v, C, M)
        amms.append(ctx.amm(cent, lut, np.float32(0.01 * (i + 1)), bias, max_n=n, tuning=named or {}))
    group = ctx.amm_group(amms)
    tiles = {a.geometry()["col_block"] for a in amms}
    fused = M % 64 == 0 or M % 48 == 0
    if named and "col_block" in named:
        fused = M % named["col_block"] == 0
    elif not named and fused and ctx.device_info()["compute_units"] == 256:
        assert len(tiles) > 1 or M % min(tiles), tiles   # (what the case is about)
    assert group.fused_cols == (len(amms) * M if fused else 0)
    x = torch.randn((min(max_n), CB * v), device="cuda", generator=torch.Generator(device="cuda").manual_seed(M))
    for n in (min(max_n), 700, 33, 1) if fused else (33,):
        want = torch.empty((n, len(amms), M), device="cuda")
        part = torch.empty((n, M), device="cuda")
        for i, a in enumerate(amms):
            torch.cuda.synchronize()
            a.run_ptr(x.data_ptr(), n, part.data_ptr())
            ctx.synchronize()
            want[:, i] = part
        if fused:
            out = torch.full((n + 1, len(amms) * M), -5.0, device="cuda")
            torch.cuda.synchronize()
            group.run_fused_ptr(x.data_ptr(), n, out.data_ptr())
            ctx.synchronize()
            assert torch.equal(out[:n], want.view(n, -1)) and bool((out[n:] == -5.0).all()), n
        else:
            with pytest.raises(pimdl.PimdlError) as e:
                group.run_fused(x[:n].cpu().numpy())
            assert e.value.code == pimdl.ERR_UNSUPPORTED
        outs = [torch.empty((n, M), device="cuda") for _ in amms]
        torch.cuda.synchronize()
        group.run_ptr(x.data_ptr(), n, [o.data_ptr() for o in outs])
        ctx.synchronize()
        assert all(torch.equal(o, want[:, i]) for i, o in enumerate(outs)), n
    group.close()
    for a in amms:
        a.close()


def test_group_conditions(ctx):
    if kernel_switches():
        pytest.skip("a kernel this test is about is switched off by the environment")
    rng = np.random.default_rng(5)
    mk = lambda K, v, C, M, kind="i8": ctx.amm(*(lambda c: (c[1], c[2]))(make_case(1, 1, K, v, C, M, kind)),
                                               None if kind == "f32" else np.float32(0.01), None, max_n=64)
    a, b = mk(128, 4, 16, 32), mk(128, 4, 16, 48)
    for bad in (mk(256, 4, 16, 32), mk(128, 2, 16, 32), mk(128, 4, 8, 32), mk(128, 4, 16, 32, "f32")):
        with pytest.raises(pimdl.PimdlError):
            ctx.amm_group([a, bad])
        bad.close()
    with pytest.raises(pimdl.PimdlError):
        ctx.amm_group([a])                       # fewer than two operators
    c40a, c40b = mk(160, 4, 16, 32), mk(160, 4, 16, 32)  # 40 codebooks: not a multiple of 32
    with pytest.raises(pimdl.PimdlError):
        ctx.amm_group([c40a, c40b])
    g = ctx.amm_group([a, b])
    with pytest.raises(pimdl.PimdlError):
        g.run(rng.standard_normal((65, 128)).astype(np.float32))  # beyond max_n
    g.close()
    for m in (a, b, c40a, c40b):
        m.close()


def test_scale_groups_from_lutgen(ctx):
    """lutgen with per-group quantisation -> operator with the same grouping: closer to the fp32 product
    than the per-tensor quantisation of the same table, and equal to the oracle on the generated table."""
    rng = np.random.default_rng(77)
    CB, C, v, M, N = 64, 16, 4, 128, 256
    cent = rng.standard_normal((CB, C, v)).astype(np.float32)
    cent[::4] *= 8.0                                     # codebooks of very different magnitude
    W = (rng.standard_normal((CB * v, M)) * 0.02).astype(np.float32)
    x = rng.standard_normal((N, CB * v)).astype(np.float32)
    lut_f, _ = ctx.lutgen(cent, W, lut_dtype=pimdl.LUT_F32)
    lut_t, s_t = ctx.lutgen(cent, W)
    lut_g, s_g = ctx.lutgen(cent, W, scale_group=1)
    assert s_g.shape == (CB,)
    idx = oracle.index_calculation(x, cent, v, threads=THREADS)
    exact = oracle.gather_f32(idx, lut_f, np.zeros(M, np.float32), threads=THREADS)
    a_t = ctx.amm(cent, lut_t, s_t, None, max_n=N)
    a_g = ctx.amm(cent, lut_g, s_g, None, max_n=N, scale_group=1)
    out_t, out_g = a_t.run(x), a_g.run(x)
    want_g = oracle.gather_i8_grouped(idx, lut_g, s_g, np.zeros(M, np.float32), 1, threads=THREADS)
    assert np.array_equal(out_g.view(np.uint32), want_g.view(np.uint32))
    err_t, err_g = np.abs(out_t - exact).mean(), np.abs(out_g - exact).mean()
    assert err_g < 0.7 * err_t, (err_g, err_t)
    a_t.close()
    a_g.close()


def test_device_pointers_and_partial_batches(ctx):
    """Inputs already resident in HBM (torch tensors), n smaller than max_n, output rows past n untouched."""
    import torch

    N, K, v, C, M = 700, 256, 4, 16, 320
    x, cent, lut, bias = make_case(41, N, K, v, C, M)
    amm = ctx.amm(cent, lut, np.float32(0.05), bias, max_n=1024)
    want = oracle.amm_cpu(x, cent, lut, bias, v, 0.05, 0.0, threads=THREADS)[0]
    xd = torch.from_numpy(x).cuda()
    od = torch.full((1024, M), -7.0, device="cuda")
    torch.cuda.synchronize()
    amm.run_ptr(xd.data_ptr(), N, od.data_ptr())
    ctx.synchronize()
    got = od.cpu().numpy()
    assert np.array_equal(got[:N].view(np.uint32), want.view(np.uint32))
    assert (got[N:] == -7.0).all()
    # a second, smaller batch through the same operator
    amm.run_ptr(xd.data_ptr(), 33, od.data_ptr())
    ctx.synchronize()
    assert np.array_equal(od.cpu().numpy()[:33].view(np.uint32), want[:33].view(np.uint32))
    amm.close()


def test_error_paths(ctx):
    cent = np.zeros((4, 16, 4), np.float32)
    lut = np.zeros((4, 16, 8), np.int8)
    with pytest.raises(pimdl.PimdlError) as e:
        ctx.amm(cent, lut, None, None)           # int8 LUT without scales
    assert e.value.code == -1
    with pytest.raises(pimdl.PimdlError) as e:           # grouped scales have no zero point
        ctx.amm(cent, lut, np.ones(2, np.float32), None, scale_group=3, lut_bias=0.5)
    assert e.value.code == -1
    amm = ctx.amm(cent, lut, np.ones(2, np.float32), None, scale_group=3, max_n=8)
    with pytest.raises(pimdl.PimdlError) as e:           # no single int32 accumulator to return
        amm.run_debug(np.zeros((4, 16), np.float32))
    assert e.value.code == -1
    amm.close()
    amm = ctx.amm(cent, lut, np.float32(1), None, max_n=8)
    with pytest.raises(pimdl.PimdlError) as e:
        amm.run(np.zeros((9, 16), np.float32))   # n > max_n
    assert e.value.code == -1
    assert amm.run(np.zeros((0, 16), np.float32)).shape == (0, 8)  # empty batch is a no-op
    amm.close()


# ---- the two-speed search: fast scores + margin test, exact replay on near ties -----------------

@pytest.mark.parametrize("v,C", [(2, 16), (4, 16), (8, 16), (4, 7), (16, 16), (4, 32), (2, 64)])
def test_search_with_exact_ties_and_degenerate_inputs(ctx, v, C):
    """Duplicate centroids (margin 0), all-zero rows, inputs equal to a centroid, tiny and huge
    magnitudes: every pair must come out as the reference's scan says, whichever path took it."""
    rng = np.random.default_rng(1000 + 10 * v + C)
    N, CB = 389, 37
    cent = rng.standard_normal((CB, C, v)).astype(np.float32)
    cent[::3, C // 2] = cent[::3, 0]                   # exact duplicates: first index must win
    cent[1::5] *= np.float32(1e-3)                     # a codebook of tiny centroids
    cent[2::7] *= np.float32(1e4)                      # and one of huge ones
    x = rng.standard_normal((N, CB, v)).astype(np.float32)
    x[::4] = 0.0
    pick = rng.integers(0, C, (N, CB))
    on = rng.random((N, CB)) < 0.3
    x[on] = cent[np.nonzero(on)[1], pick[on]]          # exactly on a centroid
    x[5::11] *= np.float32(1e5)
    x = x.reshape(N, CB * v)
    want = oracle.index_calculation(x, cent, v, threads=THREADS)
    amm = ctx.amm(cent, np.zeros((CB, C, 4), np.int8), np.float32(1.0), None, max_n=N)
    got = amm.index_calculation(x)
    assert np.array_equal(got, want), f"{(got != want).sum()} of {got.size} differ"
    amm.close()


@pytest.mark.parametrize("v,C", [(8, 16), (4, 16), (8, 32), (4, 32), (4, 20), (8, 12), (4, 5), (8, 8), (2, 16)])
def test_search_with_a_few_near_ties_per_wave(ctx, v, C):
    """One (token, codebook) pair in about 400 sits midway between two centroids, the others are ordinary: a wave
    then has one or two lanes to replay exactly, which it does lane by lane with all its lanes (many at once take
    another path, covered by the dense cases above).  Both token tiles of the search, a ragged batch, a codebook
    count that leaves the last codebook tile partly empty; every index against the reference's scan."""
    rng = np.random.default_rng(3000 + 10 * v + C)
    N, CB = 1500, 37
    cent = rng.standard_normal((CB, C, v)).astype(np.float32)
    x = rng.standard_normal((N, CB, v)).astype(np.float32)
    on = rng.random((N, CB)) < 1.0 / 400
    a = rng.integers(0, C, (N, CB))
    b = (a + 1 + rng.integers(0, C - 1, (N, CB))) % C
    cbi = np.nonzero(on)[1]
    mid = (cent[cbi, a[on]] + cent[cbi, b[on]]) * np.float32(0.5)
    x[on] = mid + rng.standard_normal(mid.shape).astype(np.float32) * np.float32(2e-7)
    x = x.reshape(N, CB * v)
    want = oracle.index_calculation(x, cent, v, threads=THREADS)
    assert (want != oracle.np_distances(x, cent).argmin(-1)).sum() > 0  # some pairs separate the scan from the true argmin
    amm = ctx.amm(cent, np.zeros((CB, C, 4), np.int8), np.float32(1.0), None, max_n=N)
    for tile in (0, 64, 128):
        amm.set_tuning(search_token_tile=tile)
        got = amm.index_calculation(x)
        assert np.array_equal(got, want), f"tile {tile}: {(got != want).sum()} of {got.size} differ"
    amm.close()


@pytest.mark.parametrize("v,C", [(2, 16), (4, 16), (8, 16), (4, 9), (2, 32), (4, 32), (8, 32), (4, 17),
                                 (2, 64), (4, 33), (8, 130), (16, 16), (32, 40)])
@pytest.mark.parametrize("size", [1e-4, 0.03, 1.0, 900.0, 1100.0, 3e4, 1e9, 1e16])
def test_search_over_the_range_of_halves(ctx, v, C, size):
    """The matrix search works on halves, whose range ends at 65504 and 6e-8: centroids and activations of one size from far below
    to far above it (codebooks with centroids beyond 1024 are searched at a scale of their own), codebooks of another size beside them in
    the same and in other tiles, activations that no half holds, an odd width; every index against the reference's scan."""
    rng = np.random.default_rng(int(4000 + 10 * v + C))
    many = C > 32 or v > 8                             # the search by groups of 32 centroids; fewer tokens take another
    N, CB = 1500 if many else 210, 37
    cent = rng.standard_normal((CB, C, v)).astype(np.float32)
    x = rng.standard_normal((N, CB, v)).astype(np.float32)
    cent[:20] *= np.float32(size)
    x[:, :20] *= np.float32(size)
    cent[3], x[:, 3] = cent[3] / np.float32(size), x[:, 3] / np.float32(size)
    x[7::50] *= np.float32(7e4)
    x[8, 30, 0], x[9, 5, v - 1] = 65504.0, -1e30
    x = x.reshape(N, CB * v)
    want = oracle.index_calculation(x, cent, v, threads=THREADS)
    amm = ctx.amm(cent, np.zeros((CB, C, 4), np.int8), np.float32(1.0), None, max_n=N)
    for tile in (0,) if many else (64, 128):
        amm.set_tuning(search_token_tile=tile)
        got = amm.index_calculation(x)
        assert np.array_equal(got, want), f"tile {tile}: {(got != want).sum()} of {got.size} differ"
    amm.close()


@pytest.mark.parametrize("v,C", [(4, 16), (2, 16), (8, 16), (4, 9), (2, 32), (4, 20), (8, 32), (2, 64), (4, 33), (8, 130), (16, 16), (32, 40)])
@pytest.mark.parametrize("length", [1e15, 1e17, 9.5e17])
def test_search_where_distances_overflow(ctx, v, C, length):
    """Finite centroids up to the longest that the matrix search takes (|c|^2 < 1e36), and rows from that length to lengths whose squared
    distances are beyond FLT_MAX for some or for all of the centroids: the reference's distances are infinite there, and its scan stays
    where it is.  Every index against that scan."""
    rng = np.random.default_rng(6000 + 10 * v + C)
    many = C > 32 or v > 8
    N, CB = 1500 if many else 330, 37
    unit = lambda a: a / np.linalg.norm(a, axis=-1, keepdims=True)
    cent = (unit(rng.standard_normal((CB, C, v))) * length * rng.uniform(0.9, 1.0, (CB, C, 1))).astype(np.float32)
    x = unit(rng.standard_normal((N, CB, v))) * rng.choice([length, 30 * length, 1.5e19, 1.8e19, 1.9e19, 2.2e19, 3.5e19], (N, CB, 1))
    x = x.astype(np.float32).reshape(N, CB * v)
    with np.errstate(all="ignore"):
        want = oracle.index_calculation(x, cent, v, threads=THREADS)
    amm = ctx.amm(cent, np.zeros((CB, C, 4), np.int8), np.float32(1.0), None, max_n=N)
    for tile in (0,) if many else (64, 128):
        amm.set_tuning(search_token_tile=tile)
        got = amm.index_calculation(x)
        assert np.array_equal(got, want), f"tile {tile}: {(got != want).sum()} of {got.size} differ"
    amm.close()


def _search_us(ctx, cent, x):
    """Shortest of several timings of the search alone."""
    import torch
    CB, C, v = cent.shape
    n = x.shape[0]
    amm = ctx.amm(cent, np.zeros((CB, C, 16), np.int8), np.float32(1.0), None, max_n=n)
    xd, out = torch.from_numpy(x).cuda(), torch.empty((n, 16), device="cuda")
    torch.cuda.synchronize()
    us = min(amm.profile(xd.data_ptr(), n, out.data_ptr(), warmup=20, iters=20)["ccs_ms"] for _ in range(5)) * 1e3
    amm.close()
    return us


@pytest.mark.parametrize("v,C", [(2, 16), (4, 16), (8, 16), (2, 32), (4, 20), (8, 32), (2, 64), (4, 33), (16, 16), (32, 40)])
@pytest.mark.parametrize("size", [2e-4, 2e-3, 0.01, 0.05, 0.3])
def test_search_of_small_centroids(ctx, v, C, size):
    """Centroids and activations whose pieces are subnormal halves, one in 100 sub-vectors close to the middle of two centroids (off it by
    up to three times the hysteresis), activations from a hundredth to a hundred times the centroids' size: every index against the reference's
    scan."""
    rng = np.random.default_rng(int(1e6 * size) + 10 * v + C)
    N, CB = 1500, 37
    cent = (rng.standard_normal((CB, C, v)) * size).astype(np.float32)
    x = (rng.standard_normal((N, CB, v)) * size).astype(np.float32)
    x[::9] *= np.float32(100)
    x[4::9] *= np.float32(0.01)
    on = rng.random((N, CB)) < 0.01
    cbi, a = np.nonzero(on)[1], rng.integers(0, C, on.sum())
    b = (a + 1 + rng.integers(0, C - 1, on.sum())) % C
    between = (cent[cbi, b] - cent[cbi, a]).astype(np.float64)
    gap = rng.uniform(-3e-6, 3e-6, (on.sum(), 1))      # of the two squared distances
    x[on] = cent[cbi, a] + between * (0.5 + gap / (2 * (between ** 2).sum(-1, keepdims=True)))
    x = x.reshape(N, CB * v)
    want = oracle.index_calculation(x, cent, v, threads=THREADS)
    amm = ctx.amm(cent, np.zeros((CB, C, 4), np.int8), np.float32(1.0), None, max_n=N)
    for tile in (0,) if C > 32 or v > 8 else (64, 128):
        amm.set_tuning(search_token_tile=tile)
        got = amm.index_calculation(x)
        assert np.array_equal(got, want), f"tile {tile}: {(got != want).sum()} of {got.size} differ"
    amm.close()


def test_search_of_small_centroids_is_not_all_replays(ctx):
    """Centroids of 0.01 in 8 dimensions: nearest and second nearest are as often within the hysteresis as they are, but what the margin
    allows for subnormal halves is in proportion to the centroids.  1.5 times the time of a launch with centroids of 1, and 1.9 to 2.1 times with an
    allowance of its own for any size."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about the library's choice")
    rng = np.random.default_rng(6100)
    cent, x = rng.standard_normal((384, 16, 8), dtype=np.float32), rng.standard_normal((8192, 3072), dtype=np.float32)
    usual, small = _search_us(ctx, cent, x), _search_us(ctx, cent * np.float32(0.01), x * np.float32(0.01))
    print(f"centroids of 1 {usual:.1f} us, of 0.01 {small:.1f}")
    assert small < 1.7 * usual, (usual, small)


@pytest.mark.parametrize("v,C", [(2, 16), (4, 16), (8, 16), (4, 32)])
def test_search_of_small_codebooks_beside_a_large_one(ctx, v, C):
    """One codebook in 16 a million times as large as the others: its neighbours are searched as they would be without it, not replayed.  The
    time of a launch in which one in 16 may be, against the same launch without a large codebook; replays of the whole tile take 2.3 to 2.8 times."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about the library's choice")
    rng = np.random.default_rng(6200 + v + C)
    N, CB = 8192, 3072 // v
    cent = rng.standard_normal((CB, C, v), dtype=np.float32)
    x = rng.standard_normal((N, CB, v), dtype=np.float32)
    plain = _search_us(ctx, cent, x.reshape(N, -1))
    cent[5::16] *= np.float32(1e6)
    x[:, 5::16] *= np.float32(1e6)
    beside = _search_us(ctx, cent, x.reshape(N, -1))
    print(f"v {v}, {C} centroids: {plain:.1f} us, beside large codebooks {beside:.1f}")
    assert beside < 1.5 * plain, (plain, beside)
    rows = np.arange(0, N, 64)
    amm = ctx.amm(cent, np.zeros((CB, C, 4), np.int8), np.float32(1.0), None, max_n=N)
    got = amm.index_calculation(x.reshape(N, -1))[rows]
    assert np.array_equal(got, oracle.index_calculation(x.reshape(N, -1)[rows], cent, v, threads=THREADS))
    amm.close()


@pytest.mark.parametrize("v,C", [(2, 16), (4, 16), (8, 16), (4, 32)])
def test_search_of_a_group_with_codebooks_of_any_size(ctx, v, C):
    """Operators that share a search read the same columns with codebooks of their own: some of each beyond 1024, others small or tiny, ties and long
    rows among the activations, so that replays read the row from memory.  Every output as of the operator alone and of the reference's scan."""
    rng = np.random.default_rng(6350 + v + C)
    N, CB, M = 700, 64, 48
    x = rng.standard_normal((N, CB, v), dtype=np.float32)
    x[::7] = 0.0
    x[3::11] *= np.float32(7e4)
    sizes = np.float32([1.0, 3e4, 1.0, 1e-3, 1e7, 30.0])
    amms, want = [], []
    for i in range(3):
        _, cent, lut, bias = make_case(6360 + i, 1, CB * v, v, C, M)
        size = sizes[rng.integers(0, len(sizes), CB)]
        cent = cent.reshape(CB, C, v) * size[:, None, None]
        cent[::5, C // 2] = cent[::5, 0]
        if i == 0:
            x *= size[:, None]
        amms.append(ctx.amm(cent, lut, np.float32(0.01), bias, max_n=N))
        want.append((cent, lut, bias))
    x = x.reshape(N, CB * v)
    group = ctx.amm_group(amms)
    for tile in (64, 128):
        for a in amms:
            a.set_tuning(search_token_tile=tile)
        tiled = ctx.amm_group(amms)              # (a group keeps the search settings that its first member has when it is created)
        for g in (group, tiled):
            for a, out, (cent, lut, bias) in zip(amms, g.run(x), want):
                idx = oracle.index_calculation(x, cent, v, threads=THREADS)
                acc = oracle.gather_i8(idx, lut, threads=THREADS)
                assert np.array_equal(out.view(np.uint32), oracle.dequant(acc, bias, CB, 0.01, 0.0, 0, threads=THREADS).view(np.uint32)), tile
                assert np.array_equal(a.index_calculation(x), idx)
        tiled.close()
    group.close()
    for a in amms:
        a.close()


@pytest.mark.parametrize("v,C", [(2, 16), (4, 16), (8, 16), (4, 32)])
def test_search_of_rows_longer_than_large_centroids(ctx, v, C):
    """Centroids of about 3000, every hundredth row of 3e5 in each dimension: far enough from a tie in every codebook but a few, and inside the range
    that halves have at the codebooks' scale.  The time against the same launch without such rows; with their replays it is 1.5 to 1.8
    times."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about the library's choice")
    rng = np.random.default_rng(6300 + v + C)
    N, CB = 8192, 3072 // v
    cent = rng.standard_normal((CB, C, v), dtype=np.float32) * np.float32(3000)
    x = rng.standard_normal((N, CB * v), dtype=np.float32) * np.float32(3000)
    plain = _search_us(ctx, cent, x)
    x[::100] = np.sign(x[::100]) * np.float32(3e5)
    beyond = _search_us(ctx, cent, x)
    print(f"v {v}, {C} centroids: {plain:.1f} us, with long rows {beyond:.1f}")
    assert beyond < 1.25 * plain, (plain, beyond)


@pytest.mark.parametrize("v,C", [(4, 16), (2, 16), (8, 16), (4, 32)])
def test_search_with_non_finite_values(ctx, v, C):
    """NaN / Inf / near-overflow values in activations and centroids take the exact path and match
    the reference's compare semantics (a NaN distance never replaces the running best)."""
    rng = np.random.default_rng(2000 + 10 * v + C)
    N, CB = 300, 40
    cent = rng.standard_normal((CB, C, v)).astype(np.float32)
    cent[3, 2, 0] = np.nan
    cent[5, 0, 1] = np.nan          # NaN in centroid 0: the scan keeps index 0
    cent[7, 4, 0] = np.inf
    cent[9, 1, :] = 3e19            # |c|^2 overflows fp32
    cent[11, 6, 0] = -np.inf
    x = rng.standard_normal((N, CB * v)).astype(np.float32)
    x[1, :] = np.nan
    x[2, 5] = np.inf
    x[3, 7] = -np.inf
    x[4, :] = 2e19
    x[6, 3] = 3e38
    with np.errstate(all="ignore"):
        want = oracle.index_calculation(x, cent, v, threads=THREADS)
    amm = ctx.amm(cent, np.zeros((CB, C, 4), np.int8), np.float32(1.0), None, max_n=N)
    got = amm.index_calculation(x)
    assert np.array_equal(got, want), f"{(got != want).sum()} of {got.size} differ"
    amm.close()


def test_matrix_core_rounding_stays_inside_the_search_margin(ctx):
    """The matrix search accepts a winner only outside an error margin that assumes every addition of
    the matrix core's chain (48 products + the initial accumulator) is within 2^-24 of the partial sum:
    51 units of 2^-24 * sum|terms| for a chain of three.  Measured on this device over 10^6 outputs with operand pieces
    of mixed magnitude, the chain stays an order of magnitude inside that."""
    worst = ctx.diag_mfma_error(1024)
    assert 0.0 < worst < 12.0, worst


def test_matrix_core_rounding_on_crafted_worst_cases(ctx):
    """Random operands are not the worst case for an accumulator.  The crafted chains add 48 equal products just
    below / above 1/2, 1 and 2 units in the last place of an accumulator of 1.0 (either sign), and products
    falling by a factor of four per slot: a sequential round-to-nearest adder loses 24 units on them, a
    truncating one up to 96.  The search margin allows 51; the device must stay below half of that."""
    worst = ctx.diag_mfma_error_crafted()
    print("crafted mfma error (units of 2^-24 * sum|terms|):", worst)
    assert 0.0 <= worst < 25.5, worst


def test_search_at_full_ffn2_shape(ctx):
    """N=8192, K=3072, v=4, 16 centroids: every index of the headline shape against the oracle,
    once with N(0,1) data and once with the reference driver's ranges."""
    for dist in ("normal", "ref"):
        x, cent, _, _ = make_case(77, 8192, 3072, 4, 16, 4, "i8", dist)
        want = oracle.index_calculation(x, cent, 4, threads=THREADS)
        amm = ctx.amm(cent, np.zeros((768, 16, 4), np.int8), np.float32(1.0), None, max_n=8192)
        got = amm.index_calculation(x)
        assert np.array_equal(got, want), f"{dist}: {(got != want).sum()} of {got.size} differ"
        amm.close()


def _random_cases(count, seed):
    rng = np.random.default_rng(seed)
    cases = []
    for i in range(count):
        v = int(rng.choice([2, 4, 8, 2, 4, 8, 3, 16]))
        C = int(rng.choice([rng.integers(2, 9), rng.integers(9, 17), rng.integers(17, 33), 16, 16, 32, 8, 64]))
        CB = int(rng.choice([rng.integers(1, 12), rng.integers(12, 80), 32, 64, 96]))
        M = int(rng.choice([rng.integers(1, 64), rng.integers(64, 420), 96, 192, 768]))
        N = int(rng.choice([rng.integers(1, 70), rng.integers(70, 700), rng.integers(700, 2600), 256, 1024]))
        kind = str(rng.choice(["i8", "i8", "i8", "f32", "grouped"]))
        cases.append((i, N, CB * v, v, C, M, kind))
    return cases


@pytest.mark.parametrize("case", _random_cases(48, 2024), ids=lambda c: "n%d_k%d_v%d_c%d_m%d_%s" % c[1:])
def test_random_shapes_against_the_oracle(ctx, case):
    """Seeded random shapes across every kernel variant (search: matrix narrow / wide, exact, generic; gather:
    one-hot, paired, byte adder, fp32 one and two tokens per lane, grouped), with a non-zero LUT bias in both
    bias modes for the int8 table."""
    i, N, K, v, C, M, kind = case
    x, cent, lut, bias = make_case(7000 + i, N, K, v, C, M, "f32" if kind == "f32" else "i8")
    CB = K // v
    want_idx = oracle.index_calculation(x, cent, v, threads=THREADS)
    if kind == "i8":
        mode = i % 2
        amm = ctx.amm(cent, lut, np.float32(0.0371), bias, max_n=N, lut_bias=0.25, bias_mode=mode)
        out, idx, acc = amm.run_debug(x)
        want_acc = oracle.gather_i8(want_idx, lut, threads=THREADS)
        assert np.array_equal(idx, want_idx)
        assert np.array_equal(acc, want_acc)
        want = oracle.dequant(want_acc, bias, CB, 0.0371, 0.25, mode, threads=THREADS)
        assert np.array_equal(out.view(np.uint32), want.view(np.uint32))
    elif kind == "f32":
        amm = ctx.amm(cent, lut, None, bias, max_n=N)
        out, idx, _ = amm.run_debug(x)
        assert np.array_equal(idx, want_idx)
        np.testing.assert_allclose(out, oracle.gather_f32(want_idx, lut, bias, threads=THREADS), rtol=1e-5,
                                   atol=1e-5 * np.sqrt(CB))
    else:
        group = 1 + i % 5
        scales = np.random.default_rng(i).uniform(1e-3, 0.1, (CB + group - 1) // group).astype(np.float32)
        amm = ctx.amm(cent, lut, scales, bias, max_n=N, scale_group=group)
        want = oracle.gather_i8_grouped(want_idx, lut, scales, bias, group, threads=THREADS)
        assert np.array_equal(amm.run(x).view(np.uint32), want.view(np.uint32))
    amm.close()


@pytest.mark.parametrize("N,CB,C,M", [
    (1, 1, 17, 1),          # one token, one codebook of a 16-codebook slice, one column of a 16-column chunk
    (63, 15, 33, 15), (65, 17, 64, 17), (129, 33, 65, 33),   # edges of token blocks, slices, rows, chunks
    (1025, 16, 32, 130),    # one token past an item, an odd number of chunks
    (2500, 48, 24, 1040), (2500, 48, 50, 1040), (2500, 32, 100, 530), (2500, 32, 250, 530),  # several item sizes
    (40000, 16, 32, 1040), (40000, 16, 64, 1040), (40000, 16, 128, 1040), (40000, 16, 256, 530),  # the widest waves
])
def test_byte_adder_edges(ctx, N, CB, C, M):
    """17 centroids and more through the byte adder: every index, accumulator and output bit of the oracle."""
    check_i8(ctx, 4200 + C + N, N, 4 * CB, 4, C, M, lut_bias=0.5, bias_mode=1)


def test_byte_adder_item_sizes(ctx):
    """The launch rule's ends: a batch that fills the chip takes eight token groups per wave, a small one a single group."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about the library's choice")
    x, cent, lut, bias = make_case(5, 40000, 64, 4, 64, 1040)
    amm = ctx.amm(cent, lut, np.float32(0.01), bias, max_n=40000)
    for n, groups in ((40000, 8), (70, 1)):
        amm.run_debug(x[:n])  # the whole batch in one launch (run cuts host buffers into chunks)
        assert amm.last_gather_kernel().split(", ")[3] == str(groups), amm.last_gather_kernel()
    amm.close()


FEW_SHAPES = [
    # N, CB, v, C, M, lut, scale_group: launches of few tokens, whose codebooks are dealt out to waves
    (1, 192, 4, 16, 3072, "i8", 0),     # one token
    (16, 40, 2, 9, 100, "i8", 0),       # the last of 16-token items; padded codebooks; a ragged column tile
    (17, 33, 4, 16, 49, "i8", 0),       # 32-token items; ragged columns of a second tile
    (33, 768, 4, 16, 768, "i8", 0),     # 64-token items, more K-steps per wave than are in flight together
    (300, 96, 4, 12, 1001, "i8", 0),    # eight waves: more items than CUs
    (5, 70, 4, 8, 100, "i8", 0),        # paired codebooks
    (300, 192, 4, 5, 768, "i8", 0),
    (1, 256, 4, 64, 1001, "i8", 0),     # byte adder
    (13, 768, 2, 17, 768, "i8", 0),
    (3, 50, 8, 256, 70, "i8", 0),
    (1, 192, 4, 16, 770, "f32", 0),     # floats: rows of 16, in 8-byte pieces (32 centroids), rows of 8
    (67, 768, 4, 8, 96, "f32", 0),
    (5, 96, 4, 32, 50, "f32", 0),
    (9, 64, 4, 130, 33, "f32", 0),
    (7, 192, 4, 16, 100, "i8", 1),      # a scale per codebook, and per 5 with a ragged last group
    (3, 193, 4, 16, 100, "i8", 5),
    (3, 64, 4, 20, 40, "i8", 7),
]


@pytest.mark.parametrize("N,CB,v,C,M,lut,group", FEW_SHAPES)
def test_launches_of_few_tokens(ctx, N, CB, v, C, M, lut, group):
    """Bit for bit the oracle's indices and output, with the guard rows behind the output untouched, and the kernel
    that takes them is the one for few tokens."""
    x, cent, table, bias = make_case(6100 + N + C, N, CB * v, v, C, M, lut)
    scales = None if lut == "f32" else np.float32(0.0123)
    if group:
        scales = np.random.default_rng(N).uniform(0.001, 0.02, (CB + group - 1) // group).astype(np.float32)
    amm = ctx.amm(cent, table, scales, bias, max_n=N, scale_group=group)
    out, idx, acc = amm.run_debug(x, want_acc=lut == "i8" and not group)
    want_idx = oracle.index_calculation(x, cent, v, threads=THREADS)
    assert np.array_equal(idx, want_idx)
    if lut == "f32":
        want = oracle.gather_f32(want_idx, table, bias, threads=THREADS)
    elif group:
        want = oracle.gather_i8_grouped(want_idx, table, scales, bias, group, threads=THREADS)
    else:
        want_acc = oracle.gather_i8(want_idx, table, threads=THREADS)
        assert np.array_equal(acc, want_acc)
        want = oracle.dequant(want_acc, bias, CB, 0.0123, 0.0, 0, threads=THREADS)
    assert np.array_equal(out.view(np.uint32), want.view(np.uint32))
    if not kernel_switches():
        assert "_few_" in amm.last_gather_kernel(), amm.last_gather_kernel()
    import torch
    guarded = torch.full((N + 3, M), -5.0, device="cuda")
    xd = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    amm.run_ptr(xd.data_ptr(), N, guarded.data_ptr())
    ctx.synchronize()
    got = guarded.cpu().numpy()
    assert np.array_equal(got[:N].view(np.uint32), want.view(np.uint32)) and (got[N:] == -5.0).all()
    amm.close()


@pytest.mark.parametrize("N,v,C", [(1, 4, 64), (5, 2, 33), (40, 8, 65), (3, 16, 128), (2, 32, 200), (70, 4, 256)])
def test_search_of_few_tokens_with_many_centroids(ctx, N, v, C):
    """A wave per (token, codebook) pair: near ties within the hysteresis in either order, repeated and zero centroids,
    NaN and infinities, codebooks that are no multiple of a workgroup's."""
    CB, M = 37, 20
    x, cent, lut, bias = make_case(7100 + N + C, N, CB * v, v, C, M)
    cent[1, :] = 0.0
    cent[2, C - 1] = cent[2, 0]
    cent[3] = cent[3, 7] + np.linspace(2e-7, 0, C, dtype=np.float32)[:, None]   # a chain of steps below the hysteresis
    cent[4] = cent[4, 7] + np.linspace(3e-4, 0, C, dtype=np.float32)[:, None]   # ... and around it
    cent[5, C // 2] = np.nan
    cent[6, 0] = np.inf
    x[:, 3 * v:5 * v] = np.tile(np.concatenate([cent[3, 7], cent[4, 7]]), (N, 1))
    x[0, 7 * v] = np.nan
    x[0, 8 * v] = np.inf
    x[0, 9 * v] = 1e30
    amm = ctx.amm(cent, lut, np.float32(0.01), bias, max_n=N)
    _, idx, _ = amm.run_debug(x)
    want = oracle.index_calculation(x, cent, v, threads=THREADS)
    assert np.array_equal(idx, want), np.argwhere(idx != want)[:8]
    amm.close()


@pytest.mark.parametrize("N,v,C,lut", [(1170, 2, 33, "i8"), (1201, 4, 64, "i8"), (3600, 4, 256, "i8"), (2000, 8, 100, "f32"), (705, 16, 65, "i8"),
                                       (200, 32, 200, "i8"), (1, 16, 8, "i8"), (65, 32, 32, "i8"), (129, 16, 16, "i8"), (63, 32, 3, "f32"),
                                       (64, 16, 32, "f32")])
def test_matrix_search_over_groups_of_centroids(ctx, N, v, C, lut):
    """More than 32 centroids, and sub-vectors of 16 and 32: ragged tiles and groups, padded codebooks, both index
    layouts; single near ties (replayed by the whole wave) and codebooks in which every token ties (lane by lane);
    NaN, infinities, magnitudes from 1e-20 to 1e20."""
    CB, M = 37, 20
    x, cent, table, bias = make_case(8100 + N + C, N, CB * v, v, C, M, lut)
    cent[1] = 0.0                                   # every token ties
    cent[2, C - 1] = cent[2, 0]                     # those nearest to the repeated centroid do
    cent[3, C // 2] = np.nan
    cent[4, 0] = np.inf
    cent[5] = cent[5, :1] + np.linspace(3e-4, 0, C, dtype=np.float32)[:, None]   # steps around the hysteresis
    x[N // 2, 2 * v:3 * v] = cent[2, 0]
    x[0, 5 * v:6 * v] = cent[5, 0]
    x[N - 1, 6 * v] = np.nan
    x[N // 3, 7 * v] = -np.inf
    x[N - 1, 8 * v:] *= np.float32(1e20)
    x[N // 4] *= np.float32(1e-20)
    amm = ctx.amm(cent, table, None if lut == "f32" else np.float32(0.01), bias, max_n=N)
    _, idx, _ = amm.run_debug(x, want_acc=False)
    want = oracle.index_calculation(x, cent, v, threads=THREADS)
    assert np.array_equal(idx, want), (int((idx != want).sum()), np.argwhere(idx != want)[:8])
    amm.close()


@pytest.mark.parametrize("N,CB,v,C,M,group", [
    (63, 32, 4, 16, 4096, 0), (500, 33, 4, 16, 500, 0), (65, 64, 2, 8, 2031, 0), (900, 96, 4, 17, 770, 0),  # 64-token workgroups
    (257, 40, 4, 16, 4100, 0), (8200, 32, 4, 7, 800, 0), (5000, 65, 4, 32, 1001, 0),                       # 256-token ones
    (600, 70, 4, 12, 100, 1), (300, 70, 4, 16, 4096, 9), (520, 41, 4, 30, 3000, 3), (900, 41, 4, 8, 64, 6)])
def test_float_tables_in_pieces(ctx, N, CB, v, C, M, group):
    """fp32 tables and scales per group of codebooks up to 32 centroids: the additions are made in ascending codebook
    order whatever the kernel, so the output is the oracle's to the bit; the last tokens and ragged columns included."""
    x, cent, table, bias = make_case(9100 + N + C, N, CB * v, v, C, M, "i8" if group else "f32")
    scales = np.random.default_rng(N).uniform(0.001, 0.02, (CB + group - 1) // group).astype(np.float32) if group else None
    amm = ctx.amm(cent, table, scales, bias, max_n=N, scale_group=group)
    out, idx, _ = amm.run_debug(x, want_acc=False)
    rows = np.unique(np.concatenate([np.arange(0, min(N, 70)), np.arange(max(0, N - 70), N),
                                     np.random.default_rng(1).choice(N, size=min(N, 100), replace=False)]))
    want_idx = oracle.index_calculation(x[rows], cent, v, threads=THREADS)
    assert np.array_equal(idx[rows], want_idx)
    want = (oracle.gather_i8_grouped(want_idx, table, scales, bias, group, threads=THREADS) if group
            else oracle.gather_f32(want_idx, table, bias, threads=THREADS))
    assert np.array_equal(out[rows].view(np.uint32), want.view(np.uint32))
    assert "_f32_rows_" in amm.last_gather_kernel(), amm.last_gather_kernel()
    amm.close()


@pytest.mark.parametrize("CB,v,C,M,group", [(48, 4, 16, 1001, 0), (7, 3, 17, 333, 2), (96, 4, 16, 1024, 1), (3, 8, 5, 6, 0), (64, 4, 64, 1537, 5)])
@pytest.mark.parametrize("ordered", [False, True])
def test_lutgen_quantisation_of_any_group(ctx, CB, v, C, M, group, ordered):
    """The int8 table and the scales are those of the fp32 table of the same call form to the bit: magnitudes per workgroup,
    entries four at a time and one by one (group boundaries that are no multiple of four), pieces through the pinned
    ring and small buffers, an all-zero group."""
    rng = np.random.default_rng(CB + M)
    cent = rng.standard_normal((CB, C, v)).astype(np.float32)
    weight = (rng.standard_normal((CB * v, M)) * 0.02).astype(np.float32)
    cbs = group or CB
    if group:
        cent[cbs:2 * cbs] = 0.0
    full, _ = ctx.lutgen(cent, weight, lut_dtype=pimdl.LUT_F32, ordered=ordered)
    if ordered:
        assert np.array_equal(full.view(np.uint32), oracle.lutgen_f32(cent, weight, threads=THREADS).view(np.uint32))
    table, scales = ctx.lutgen(cent, weight, scale_group=group, ordered=ordered)
    for g in range((CB + cbs - 1) // cbs):
        part = full[g * cbs:(g + 1) * cbs]
        s = np.abs(part).max() / np.float32(127)
        s = s if s > 0 else np.float32(1)
        assert scales[g] == s
        assert np.array_equal(table[g * cbs:(g + 1) * cbs], np.rint(np.clip(part / s, -128, 127)).astype(np.int8))


@pytest.mark.parametrize("CB,v,C,M,group", [(1, 2, 2, 3, 0), (64, 4, 256, 1024, 0), (130, 2, 40, 3001, 1), (61, 8, 33, 2083, 7), (256, 4, 64, 1028, 0)])
def test_lutgen_through_several_pieces_of_the_ring(ctx, CB, v, C, M, group):
    """Weights and tables from less than a piece of the pinned ring to more than its slots hold, whole and ragged pieces, rows that are and
    that are no multiple of 16 bytes: the float table is the matrix product's (1e-5 of the root mean square: v products of N(0, 1) x
    N(0, 0.02) in fp32), the int8 table and the scales are that table's to the bit, twice in a row through the same slots."""
    rng = np.random.default_rng(CB * M)
    cent = rng.standard_normal((CB, C, v)).astype(np.float32)
    weight = (rng.standard_normal((CB * v, M)) * 0.02).astype(np.float32)
    cbs = group or CB
    for _ in range(2):
        full, _ = ctx.lutgen(cent, weight, lut_dtype=pimdl.LUT_F32)
        want = np.matmul(cent, weight.reshape(CB, v, M))
        assert np.abs(full - want).max() <= 1e-5 * np.sqrt(np.mean(np.square(want, dtype=np.float64)))
        table, scales = ctx.lutgen(cent, weight, scale_group=group)
        for g in range((CB + cbs - 1) // cbs):
            part = full[g * cbs:(g + 1) * cbs]
            assert scales[g] == np.abs(part).max() / np.float32(127)
            assert np.array_equal(table[g * cbs:(g + 1) * cbs], np.rint(np.clip(part / scales[g], -128, 127)).astype(np.int8))
        cent = cent[::-1].copy()


def test_lutgen_takes_device_memory_for_its_own_scratch_only(ctx):
    """A context's first table construction, of a few KB and of 12 MB of weight: device memory for centroids, weight, table and magnitudes, and
    none for the pinned ring's chunks of a batch (32 MB that no table construction reads)."""
    import torch
    rng = np.random.default_rng(31)
    for K, M, v, C in ((64, 64, 4, 16), (1024, 3072, 4, 16)):
        cent, weight = rng.standard_normal((K // v, C, v), dtype=np.float32), rng.standard_normal((K, M), dtype=np.float32)
        want = ctx.lutgen(cent, weight)          # (the kernels' code objects are on the device)
        fresh = pimdl.Context(0)
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        got = fresh.lutgen(cent, weight)
        used = before - torch.cuda.mem_get_info()[0]
        scratch = 4 * (cent.size + weight.size + K // v * ((M + 255) // 256)) + want[0].size
        assert used <= scratch + (4 << 20), (used, scratch)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        x = rng.standard_normal((3000, K), dtype=np.float32)   # a batch from host buffers has them, after table construction too
        amm = fresh.amm(cent, got[0], got[1], None, max_n=3000)
        idx = oracle.index_calculation(x[:50], cent, v, threads=THREADS)
        out = amm.run(x)
        assert np.array_equal(out[:50], oracle.dequant(oracle.gather_i8(idx, got[0], threads=THREADS), np.zeros(M, np.float32), K // v, float(got[1][0]), 0.0, 0, threads=THREADS))
        assert np.array_equal(fresh.lutgen(cent[::-1].copy(), weight)[0], ctx.lutgen(cent[::-1].copy(), weight)[0])
        amm.close()
        fresh.close()


@pytest.mark.parametrize("N,CB,v,C,lut", [(9000, 1, 2, 256, "f32"), (5000, 2, 8, 100, "f32"), (700, 31, 4, 65, "i8"), (900, 33, 2, 130, "f32"),
                                          (300, 33, 16, 64, "i8"), (8200, 1, 4, 200, "i8"), (3, 70, 2, 40, "f32")])
def test_search_of_few_pairs_writes_the_padding_too(ctx, N, CB, v, C, lut):
    """A wave per (token, codebook) pair, several tokens per wave: the indices are the oracle's, and those of the padded codebooks are
    zero (a float table would add whatever lies behind its rows)."""
    x, cent, table, bias = make_case(8800 + N + CB, N, CB * v, v, C, 20, lut)
    amm = ctx.amm(cent, table, None if lut == "f32" else np.float32(0.01), bias, max_n=N)
    other = ctx.amm(cent[::-1], table, None if lut == "f32" else np.float32(0.01), bias, max_n=N)
    other.run_debug(x + np.float32(1), want_acc=False)   # leaves other indices in the context's scratch
    out, idx, _ = amm.run_debug(x, want_acc=False)
    want_idx = oracle.index_calculation(x, cent, v, threads=THREADS)
    assert np.array_equal(idx, want_idx)
    want = (oracle.gather_f32(want_idx, table, bias, threads=THREADS) if lut == "f32"
            else oracle.dequant(oracle.gather_i8(want_idx, table, threads=THREADS), bias, CB, 0.01, 0.0, 0, threads=THREADS))
    assert np.array_equal(out.view(np.uint32), want.view(np.uint32))
    amm.close()
    other.close()


@pytest.mark.parametrize("v,C", [(2, 64), (2, 256), (8, 128)])
def test_search_of_one_codebook_takes_no_longer_than_that_of_eight(ctx, v, C):
    """The search's launch rule prices what its waves do: a codebook among 31 padded ones is one codebook."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about the library's choice")
    import torch
    for N in (20000, 50000):
        us = []
        for CB in (1, 8):
            _, cent, table, bias = make_case(CB, 1, CB * v, v, C, 16)
            amm = ctx.amm(cent, table, np.float32(0.01), bias, max_n=N)
            x, y = torch.randn(N, CB * v, device="cuda"), torch.empty(N, 16, device="cuda")
            torch.cuda.synchronize()
            us.append(min(amm.profile(x.data_ptr(), N, y.data_ptr(), warmup=5, iters=20)["ccs_ms"] for _ in range(5)) * 1e3)
            amm.close()
        assert us[0] < 1.2 * us[1] + 1, (N, us)


def test_tuning_of_an_operator_the_library_gave_to_the_byte_adder(ctx):
    """17..32 centroids, created without settings: a setting of the sparse kernel takes effect (as it does at creation), what
    get_tuning reports is accepted by set_tuning and by the creation of another operator, no settings lead back to the byte adder."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about the library's choice")
    N, CB, v, C, M = 700, 41, 4, 27, 200
    x, cent, lut, bias = make_case(61, N, CB * v, v, C, M)
    amm = ctx.amm(cent, lut, np.float32(0.01), bias, max_n=N)
    want = oracle.amm_cpu(x, cent, lut, bias, v, 0.01, 0.0, threads=THREADS)[0]

    def run(op):
        assert np.array_equal(op.run(x).view(np.uint32), want.view(np.uint32))
        return op.last_gather_kernel()

    assert run(amm).startswith("gather_i8_kernel") and amm.tuning()["gather_kernel"] == pimdl.GATHER_ROWS
    untuned = amm.tuning()
    for setting in ({"token_item": 128}, {"token_item": 256}, {"cb_per_slice": 16}, {"gather_kernel": pimdl.GATHER_SPARSE},
                    {"token_item": 128, "xcd_col_split": 2, "search_kernel": 1}, {}, {"xcd_col_split": pimdl.XCD_PLAIN}, {"search_kernel": 3}):
        amm.set_tuning(**setting)
        sparse = any(k != "search_kernel" for k in setting)
        kernel, tuned = run(amm), amm.tuning()
        assert kernel.startswith("gather_sparse_kernel" if sparse else "gather_i8_kernel"), (setting, kernel)
        assert tuned["gather_kernel"] == (pimdl.GATHER_SPARSE if sparse else pimdl.GATHER_ROWS)
        assert all(tuned[k] == val for k, val in setting.items())
        if "token_item" in setting:
            assert amm.geometry()["tokens_per_wg"] == setting["token_item"]
        same = ctx.amm(cent, lut, np.float32(0.01), bias, max_n=N, tuning=tuned)
        assert same.tuning() == tuned and run(same) == kernel
        same.close()
        amm.set_tuning(**tuned)
        assert amm.tuning() == tuned and run(amm) == kernel
    for bad in ({"token_item": 100}, {"token_item": 512}, {"cb_per_slice": 64}, {"gather_kernel": pimdl.GATHER_ONEHOT},
                {"gather_kernel": pimdl.GATHER_ROWS, "token_item": 128}, {"gather_kernel": pimdl.GATHER_SPARSE, "col_block": 80}):
        before = amm.tuning()
        with pytest.raises(pimdl.PimdlError) as e:
            amm.set_tuning(**bad)
        assert e.value.code == pimdl.ERR_INVALID and amm.tuning() == before, bad
    amm.set_tuning()
    assert amm.tuning() == untuned
    amm.set_tuning(token_item=128)
    amm.run(x[:1])   # one token: the setting is the sparse kernel's
    assert amm.last_gather_kernel().startswith("gather_sparse_kernel")
    amm.set_tuning()
    amm.run(x[:1])
    assert "_few_" in amm.last_gather_kernel()
    amm.close()


@pytest.mark.parametrize("N,C,M,home", [(9856, 16, 1280, 48), (2304, 16, 768, 64), (8200, 8, 1001, 48), (600, 11, 128, 48)])
def test_settings_that_one_column_tile_has(ctx, N, C, M, home):
    """Slices of 64 codebooks are the 48-column tile's, and eight waves with slices of 16 the 64-column one's: an operator whose tile the library
    chooses has either, whichever tile suits it alone, when it is created and afterwards; a tile that the caller names does not change."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about the library's choice")
    import torch
    CB, v = 128, 2
    x, cent, lut, bias = make_case(6400 + M, 300, CB * v, v, C, M)
    want = oracle.amm_cpu(x, cent, lut, bias, v, 0.01, 0.0, threads=THREADS)[0]
    local = pimdl.Context(0)

    def make(**tuning):
        return local.amm(cent, lut, np.float32(0.01), bias, max_n=N, tuning=tuning)

    def check(op, block, slices=0):
        assert op.geometry()["col_block"] == block == op.tuning()["col_block"]
        assert np.array_equal(op.run(x).view(np.uint32), want.view(np.uint32))
        if slices:
            assert "<%d, 4, %d, 8" % (block // 16, slices) in op.last_gather_kernel(), op.last_gather_kernel()

    amm = make(**({"gather_kernel": pimdl.GATHER_SPARSE} if C == 8 else {}))
    if local.device_info()["compute_units"] == 256:
        check(amm, home)
    home = amm.geometry()["col_block"]
    stream = torch.cuda.Stream()
    xd, out = torch.from_numpy(x).cuda(), torch.empty(300, M, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        local.set_stream(stream.cuda_stream)
        amm.run_ptr(xd.data_ptr(), 300, out.data_ptr())
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
            amm.run_ptr(xd.data_ptr(), 300, out.data_ptr())
            with pytest.raises(pimdl.PimdlError):   # the other table cannot be laid out here
                amm.set_tuning(**({"token_item": 512, "cb_per_slice": 16} if home == 48 else {"token_item": 256, "cb_per_slice": 64}))
            assert amm.geometry()["col_block"] == home
    local.set_stream(None)
    for _ in range(2):
        for token_item, slices, block in ((512, 16, 64), (512, 64, 48), (512, 32, home), (256, 64, 48), (128, 32, home), (0, 0, home)):
            amm.set_tuning(token_item=token_item, cb_per_slice=slices)
            assert amm.tuning()["token_item"] == token_item and amm.tuning()["cb_per_slice"] == slices
            check(amm, block, slices if token_item == 512 else 0)
            tuned = amm.tuning()
            amm.set_tuning(**tuned)
            assert amm.tuning() == tuned
            out.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(out.cpu().numpy(), want), (token_item, slices)
    for bad in ({"token_item": 512, "cb_per_slice": 48}, {"token_item": 128, "cb_per_slice": 64}, {"col_block": 112 - home}):
        with pytest.raises(pimdl.PimdlError) as e:
            amm.set_tuning(**bad)
        assert e.value.code == pimdl.ERR_INVALID and amm.geometry()["col_block"] == home
    amm.close()
    kernel = {"gather_kernel": pimdl.GATHER_SPARSE} if C == 8 else {}
    for token_item, slices, block in ((512, 16, 64), (512, 64, 48), (256, 64, 48), (512, 32, home)):
        amm = make(token_item=token_item, cb_per_slice=slices, **kernel)
        check(amm, block, slices if token_item == 512 else 0)
        amm.close()
    for token_item, slices, block in ((512, 16, 48), (512, 64, 64), (256, 64, 64)):
        with pytest.raises(pimdl.PimdlError) as e:
            make(token_item=token_item, cb_per_slice=slices, col_block=block, **kernel)
        assert e.value.code == pimdl.ERR_INVALID
    local.close()


def test_a_graph_captured_before_a_change_of_tables_replays(ctx):
    """A captured run holds the address of the table it was captured with."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about the library's choice")
    import torch
    N, CB, v, C, M = 600, 32, 4, 32, 192
    x, cent, lut, bias = make_case(62, N, CB * v, v, C, M)
    local = pimdl.Context(0)
    amm = local.amm(cent, lut, np.float32(0.01), bias, max_n=N)
    stream = torch.cuda.Stream()
    xd, out, eager = torch.from_numpy(x).cuda(), torch.empty(N, M, device="cuda"), torch.empty(N, M, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        local.set_stream(stream.cuda_stream)
        amm.run_ptr(xd.data_ptr(), N, out.data_ptr())
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
            amm.run_ptr(xd.data_ptr(), N, out.data_ptr())
            with pytest.raises(pimdl.PimdlError):   # the other table cannot be laid out here
                amm.set_tuning(token_item=128)
        want = oracle.amm_cpu(x, cent, lut, bias, v, 0.01, 0.0, threads=THREADS)[0]
        for setting in ({"token_item": 128}, {}, {"token_item": 256}, {}):
            amm.set_tuning(**setting)
            eager.zero_()
            out.zero_()
            amm.run_ptr(xd.data_ptr(), N, eager.data_ptr())
            graph.replay()
            stream.synchronize()
            assert np.array_equal(eager.cpu().numpy(), want) and np.array_equal(out.cpu().numpy(), want), setting
    local.set_stream(None)
    amm.close()
    local.close()


@pytest.mark.parametrize("M", [48, 96, 720, 1056, 64, 320])
@pytest.mark.parametrize("settings", [({}, {}, {}), ({}, {"token_item": 128}, {}), ({"token_item": 128}, {"token_item": 128}, {}),
                                      ({"gather_kernel": pimdl.GATHER_SPARSE}, {}, {"token_item": 256}), ({"token_item": 256},) * 3])
def test_operators_side_by_side_of_17_to_32_centroids(ctx, M, settings):
    """One gather launch over operators whose widths are multiples of 48 or 64, whichever kernel each of them runs on: a few
    tokens and many, every column bit for bit that of the operator alone."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about the library's choice")
    N, CB, v, C = 2100, 32, 4, 20
    x = make_case(70, N, CB * v, v, C, M)[0]
    amms = []
    for i, setting in enumerate(settings):
        _, cent, lut, bias = make_case(71 + i, 1, CB * v, v, C, M)
        created = {k: val for k, val in setting.items() if k == "gather_kernel"}
        if created:
            created["col_block"] = 48 if M % 64 else 64
        amms.append(ctx.amm(cent, lut, np.float32(0.01 * (i + 1)), bias, max_n=N, tuning=created))
        if not created:
            amms[i].set_tuning(**setting)
    group = ctx.amm_group(amms)
    one_table = not any("gather_kernel" in s for s in settings) and not all(settings)
    if one_table:   # the byte adder's, whose columns are dealt out sixteen at a time
        assert group.fused_cols == 3 * M
    elif all(s == settings[0] for s in settings):
        assert (group.fused_cols > 0) == (M % amms[0].geometry()["col_block"] == 0)
    for n in (N, 40):
        want = np.concatenate([a.run(x[:n]) for a in amms], axis=1)
        assert np.array_equal(np.concatenate(group.run(x[:n]), axis=1).view(np.uint32), want.view(np.uint32))
        if group.fused_cols:
            assert np.array_equal(group.run_fused(x[:n]).view(np.uint32), want.view(np.uint32))
    group.close()
    for a in amms:
        a.close()


@pytest.mark.parametrize("C,v", [(16, 4), (7, 2), (32, 4)])
@pytest.mark.parametrize("order", [("rows", "f32", "scales"), ("f32", "rows"), ("scales", "rows", "rows")])
def test_byte_adder_and_float_tables_in_one_group(ctx, C, v, order):
    """Operators created for the byte adder share a search with tables resident as floats, whose index rows lie differently;
    those on the matrix-core gathers do not."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about what the caller names")
    N, CB = 333, 64
    x = make_case(80, N, CB * v, v, C, 1)[0]

    def make(kind, i):
        M = (96, 50, 130)[i]
        _, cent, table, bias = make_case(81 + i, 1, CB * v, v, C, M, "f32" if kind == "f32" else "i8")
        if kind == "scales":
            return ctx.amm(cent, table, np.linspace(0.001, 0.02, CB, dtype=np.float32), bias, max_n=N, scale_group=1)
        return ctx.amm(cent, table, None if kind == "f32" else np.float32(0.01), bias, max_n=N,
                       tuning={"gather_kernel": pimdl.GATHER_ROWS} if kind == "rows" else {})

    amms = [make(kind, i) for i, kind in enumerate(order)]
    group = ctx.amm_group(amms)
    assert group.fused_cols == 0
    for n in (N, 1, 64, 65):
        for a, o in zip(amms, group.run(x[:n])):
            assert np.array_equal(o.view(np.uint32), a.run(x[:n]).view(np.uint32)), (n, a.last_gather_kernel())
    group.close()
    default = make("i8", 0)   # the matrix-core gather, or the byte adder by the library's own choice
    with pytest.raises(pimdl.PimdlError) as e:
        ctx.amm_group([amms[0], default])
    assert e.value.code == pimdl.ERR_UNSUPPORTED
    for a in amms + [default]:
        a.close()


@pytest.mark.parametrize("C", [8, 16, 20, 64])
@pytest.mark.parametrize("N,CB,M", [(1500, 33, 200), (200, 40, 1030), (9000, 16, 130)])
def test_column_width_of_the_byte_adder(ctx, C, N, CB, M):
    """A width that the caller names is the width of the launch's items, at creation and on the operator; without one the launch
    picks, get_tuning says so, and an operator created with what it says launches the same."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about what the caller names")
    v = 2
    x, cent, lut, bias = make_case(90 + C, N, CB * v, v, C, M)
    want = oracle.amm_cpu(x, cent, lut, bias, v, 0.01, 0.0, threads=THREADS)[0]
    make = lambda **t: ctx.amm(cent, lut, np.float32(0.01), bias, max_n=N, tuning=t)

    def kernel(op):
        assert np.array_equal(op.run_debug(x)[0].view(np.uint32), want.view(np.uint32))
        name = op.last_gather_kernel()
        assert name.startswith("gather_i8_kernel<"), name
        return name

    rows = {"gather_kernel": pimdl.GATHER_ROWS}
    free = make(**rows)
    picked = kernel(free)
    assert free.tuning()["col_block"] == 0
    again = make(**free.tuning())
    assert kernel(again) == picked and again.tuning() == free.tuning()
    for width in (48, 64):
        hinted = make(**rows, col_block=width)
        assert kernel(hinted).split(", ")[1] == str(width // 16)
        assert hinted.tuning()["col_block"] == hinted.geometry()["col_block"] == width
        if C > 8:   # (up to 8 centroids the width given at creation is not binding)
            with pytest.raises(pimdl.PimdlError):
                hinted.set_tuning(col_block=112 - width)
            hinted.set_tuning()
            assert kernel(hinted).split(", ")[1] == str(width // 16)
        free.set_tuning(col_block=width)
        assert kernel(free) == kernel(hinted) and free.tuning() == hinted.tuning()
        hinted.close()
    free.set_tuning()
    assert kernel(free) == picked
    with pytest.raises(pimdl.PimdlError):
        free.set_tuning(col_block=96)
    free.close()
    again.close()


@pytest.mark.parametrize("C", [100, 200])
def test_wide_tables_have_one_column_width(ctx, C):
    x, cent, lut, bias = make_case(95, 300, 64, 4, C, 50)
    amm = ctx.amm(cent, lut, np.float32(0.01), bias, max_n=300)
    want = amm.run(x)
    for t in ({"col_block": 32}, amm.tuning(), {}):
        amm.set_tuning(**t)
        assert np.array_equal(amm.run(x), want)
    again = ctx.amm(cent, lut, np.float32(0.01), bias, max_n=300, tuning=amm.tuning())
    assert np.array_equal(again.run(x), want) and again.tuning() == amm.tuning()
    with pytest.raises(pimdl.PimdlError):
        amm.set_tuning(col_block=64)
    amm.close()
    again.close()


def test_the_reported_gather_kernel_is_a_kernel_of_the_library(ctx):
    """What last_gather_kernel names is what a profile of the launch lists: a kernel of the library, template arguments included
    (the sparse gather's last one is left out where it is 1)."""
    import subprocess
    listed = subprocess.run(["nm", "-C", pimdl.LIB_PATH], check=True, capture_output=True, text=True).stdout
    kernels = {line.split("(anonymous namespace)::", 1)[1].split(">(")[0] + ">" for line in listed.splitlines() if "::gather_" in line and ">(" in line}
    seen = set()
    for N, CB, v, C, M, lut, group in FEW_SHAPES + [(3000, 64, 4, C, 768, lut, g) for C in (8, 16, 32, 64, 200)
                                                    for lut, g in (("i8", 0), ("f32", 0), ("i8", 4))]:
        x, cent, table, _ = make_case(N + C, N, CB * v, v, C, M, lut)
        scales = None if lut == "f32" else np.full((CB + group - 1) // group, 0.01, np.float32) if group else np.float32(0.01)
        amm = ctx.amm(cent, table, scales, None, max_n=N, scale_group=group)
        amm.run(x)
        name = amm.last_gather_kernel()
        assert name in kernels or name[:-1] + ", 1>" in kernels, name
        seen.add(name.split("<")[0])
        amm.close()
    if not kernel_switches():
        assert {"gather_sparse_few_kernel", "gather_onehot_few_kernel", "gather_i8_few_kernel", "gather_f32_few_kernel", "gather_sparse_kernel",
                "gather_i8_kernel", "gather_f32_rows_kernel", "gather_f32_kernel"} <= seen, seen


@pytest.mark.parametrize("kernel,C,widths", [("ONEHOT", 16, (48, 64, 96)), ("ONEHOT", 5, (48, 64)), ("SPARSE", 16, (48, 64, 96)),
                                             ("SPARSE", 7, (64,)), ("SPARSE", 20, (48, 64, 96))])
@pytest.mark.parametrize("N,CB,M", [(255, 6, 63), (1000, 64, 130), (700, 33, 1001), (513, 32, 52), (257, 96, 1)])
def test_matrix_core_gathers_at_ragged_sizes(ctx, kernel, C, widths, N, CB, M):
    """The gathers of large launches, kept on small ones by naming their items: ragged token tiles, ragged and odd widths (scalar
    stores), padded codebooks, every item size and slice depth; indices, accumulators, output bits and the rows behind the output."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about what the caller names")
    import torch
    v = 4
    x, cent, lut, bias = make_case(9900 + N + C, N, CB * v, v, C, M)
    want, want_idx, want_acc = oracle.amm_cpu(x, cent, lut, bias, v, 0.0123, 0.0, threads=THREADS)
    xd = torch.from_numpy(x).cuda()
    entries = (CB + 31) // 32 * 32 * (2 if C > 16 else 1)   # table entries of 16 slots
    for width in widths:
        amm = ctx.amm(cent, lut, np.float32(0.0123), bias, max_n=N, tuning={"gather_kernel": getattr(pimdl, "GATHER_" + kernel), "col_block": width})
        items = [{"token_item": 128}, {"token_item": 256}, {"token_item": 256, "cb_per_slice": 16}]
        if kernel == "SPARSE" and C <= 16:
            items += [{"token_item": 512}]
            if width == 48 and entries % 64 == 0:
                items += [{"token_item": t, "cb_per_slice": 64} for t in (256, 512)]   # (256: the split between the waves of a SIMD)
        for item in items:
            amm.set_tuning(**item)
            out, idx, acc = amm.run_debug(x)
            name = amm.last_gather_kernel()
            assert name.startswith(f"gather_{kernel.lower()}_kernel<{width // 16}, "), (name, item)
            assert amm.geometry()["tokens_per_wg"] == item["token_item"], (name, item)
            assert np.array_equal(idx, want_idx) and np.array_equal(acc, want_acc), (name, item)
            assert np.array_equal(out.view(np.uint32), want.view(np.uint32)), (name, item)
            guarded = torch.full((N + 3, M), -5.0, device="cuda")
            torch.cuda.synchronize()
            amm.run_ptr(xd.data_ptr(), N, guarded.data_ptr())
            ctx.synchronize()
            got = guarded.cpu().numpy()
            assert np.array_equal(got[:N].view(np.uint32), want.view(np.uint32)) and (got[N:] == -5.0).all(), (name, item)
        amm.close()


@pytest.mark.parametrize("N,CB,v,C,M", [(1, 192, 4, 16, 3072), (2, 96, 8, 16, 2300), (1, 256, 2, 16, 768), (2, 128, 4, 9, 100), (1, 1, 4, 16, 1),
                                        (2, 3, 2, 1, 17), (1, 97, 8, 16, 4000), (2, 33, 4, 13, 63), (1, 200, 4, 10, 1000)])
def test_one_launch_for_one_or_two_tokens(ctx, N, CB, v, C, M):
    """Search and gather in one launch: the output bits of the oracle and of the two launches, with near ties, repeated centroids, NaN and
    infinities in the row, rows that are only 4-byte aligned, and through the allocation-free entry; nothing behind the output."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape")
    import torch
    x, cent, lut, bias = make_case(8100 + N + CB, N, CB * v, v, C, M)
    rng = np.random.default_rng(CB + C)
    if C > 2:
        cent[::3, C // 2] = cent[::3, 0]
        cent[1::3, C - 1] = cent[1::3, 1] + np.float32(3e-7)
    xv = x.reshape(N, CB, v)
    near = cent[np.arange(CB), rng.integers(0, C, (N, CB))]
    pick = rng.random((N, CB)) < 0.4
    xv[pick] = near[pick] + rng.choice([0.0, 1e-4, 5e-4], (int(pick.sum()), 1)).astype(np.float32)
    xv[rng.random((N, CB)) < 0.02] = np.nan
    xv[rng.random((N, CB)) < 0.02] = np.inf
    want = oracle.amm_cpu(x, cent, lut, bias, v, 0.0123, 0.0, threads=THREADS)[0]
    amm = ctx.amm(cent, lut, np.float32(0.0123), bias, max_n=8, tuning={"gather_kernel": pimdl.GATHER_SPARSE})
    two = amm.run_debug(x)[0]
    assert "_fused_" not in amm.last_gather_kernel()
    assert np.array_equal(two.view(np.uint32), want.view(np.uint32))
    for shift in (0, 1):
        xd = torch.empty(N * CB * v + shift, device="cuda")[shift:]
        xd.copy_(torch.from_numpy(x.reshape(-1)).cuda())
        for run in (amm.run_ptr, amm.run_noalloc_ptr):
            out = torch.full((N + 1, M), -5.0, device="cuda")
            torch.cuda.synchronize()
            run(xd.data_ptr(), N, out.data_ptr())
            ctx.synchronize()
            got = out.cpu().numpy()
            if ctx.device_info()["compute_units"] == 256:
                assert amm.last_gather_kernel().startswith(f"gather_sparse_few_fused_kernel<{v}, "), amm.last_gather_kernel()
            assert np.array_equal(got[:N].view(np.uint32), want.view(np.uint32)) and (got[N:] == -5.0).all(), (shift, run.__name__)
    amm.close()


@pytest.mark.parametrize("N,v,lut_bias,mode,with_bias,act", [(1, 4, 0.25, 0, True, 0), (2, 8, 0.25, 1, True, 0), (1, 2, -0.125, 1, False, 0), (2, 4, 0.0, 0, False, 0),
                                                             (1, 8, 0.25, 1, True, 1), (2, 2, 0.0, 0, False, 1)])
def test_epilogue_of_one_launch(ctx, N, v, lut_bias, mode, with_bias, act):
    """Bias or none, the table's own bias once or per codebook, GELU: the bits of the two launches, and without GELU the oracle's."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape")
    import torch
    CB, C, M = 75, 16, 500
    x, cent, lut, bias = make_case(8300 + N + v, N, CB * v, v, C, M)
    bias = bias if with_bias else None
    amm = ctx.amm(cent, lut, np.float32(0.0371), bias, max_n=8, lut_bias=lut_bias, bias_mode=mode,
                  activation=pimdl.ACT_GELU_TANH if act else pimdl.ACT_NONE)
    two, idx, acc = amm.run_debug(x)
    if not act:
        want = oracle.dequant(acc, np.zeros(M, np.float32) if bias is None else bias, CB, 0.0371, lut_bias, mode, threads=THREADS)
        assert np.array_equal(two.view(np.uint32), want.view(np.uint32))
    xd, out = torch.from_numpy(x).cuda(), torch.full((N + 1, M), -5.0, device="cuda")
    torch.cuda.synchronize()
    amm.run_ptr(xd.data_ptr(), N, out.data_ptr())
    ctx.synchronize()
    if ctx.device_info()["compute_units"] == 256:
        assert "_fused_" in amm.last_gather_kernel(), amm.last_gather_kernel()
    got = out.cpu().numpy()
    assert np.array_equal(got[:N].view(np.uint32), two.view(np.uint32)) and (got[N:] == -5.0).all()
    amm.close()


@pytest.mark.parametrize("N", [1, 2, 3])
def test_profile_times_the_pass_that_a_run_makes(ctx, N):
    """total_ms is of the launches of pimdl_amm_run, one or two; the last of them is what the operator names afterwards."""
    import torch
    x, cent, lut, bias = make_case(930 + N, N, 512, 4, 16, 300)
    want = oracle.amm_cpu(x, cent, lut, bias, 4, 0.0123, 0.0, threads=THREADS)[0]
    amm = ctx.amm(cent, lut, np.float32(0.0123), bias, max_n=4)
    xd, out = torch.from_numpy(x).cuda(), torch.empty((N, 300), device="cuda")
    torch.cuda.synchronize()
    t = amm.profile(xd.data_ptr(), N, out.data_ptr(), warmup=2, iters=3)
    profiled = amm.last_gather_kernel()
    assert all(ms > 0 for ms in t.values())
    assert np.array_equal(out.cpu().numpy().view(np.uint32), want.view(np.uint32))
    amm.run_ptr(xd.data_ptr(), N, out.data_ptr())
    ctx.synchronize()
    assert profiled == amm.last_gather_kernel()
    if ctx.device_info()["compute_units"] == 256 and not kernel_switches():
        assert ("_fused_" in profiled) == (N <= 2), profiled
    amm.close()


@pytest.mark.parametrize("N", [1, 2, 3])
@pytest.mark.parametrize("K,M,v,shift", [(512, 512, 4, 0), (256, 256, 2, 0), (256, 256, 2, 100), (512, 512, 8, -300), (256, 700, 4, 255), (512, 100, 4, 30),
                                         (256, 256, 4, -1), (256, 700, 4, None), (512, 100, 4, None)])
def test_output_that_lies_on_the_input(ctx, N, K, M, v, shift):
    """The output's first float `shift` floats behind the input's: every row is searched as it was before the call, for one and two tokens too.
    (None: right behind the input's last float, which one launch bears.)"""
    import torch
    x, cent, lut, bias = make_case(910 + N + K, N, K, v, 16, M)
    want = oracle.amm_cpu(x, cent, lut, bias, v, 0.0123, 0.0, threads=THREADS)[0]
    amm = ctx.amm(cent, lut, np.float32(0.0123), bias, max_n=4)
    at = N * K if shift is None else shift
    start = 1000  # of the input in the buffer
    for run in (amm.run_ptr, amm.run_noalloc_ptr):
        buf = torch.full((start + N * (K + M) + 1000,), -5.0, device="cuda")
        buf[start:start + N * K] = torch.from_numpy(x.reshape(-1)).cuda()
        torch.cuda.synchronize()
        run(buf.data_ptr() + 4 * start, N, buf.data_ptr() + 4 * (start + at))
        ctx.synchronize()
        got = buf[start + at:start + at + N * M].cpu().numpy().reshape(N, M)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), run.__name__
        if ctx.device_info()["compute_units"] == 256 and not kernel_switches():
            assert ("_fused_" in amm.last_gather_kernel()) == (shift is None and N <= 2), amm.last_gather_kernel()
    amm.close()


@pytest.mark.parametrize("N,CB,v,C", [(1, 1, 4, 16), (3, 33, 4, 9), (64, 70, 2, 16), (230, 192, 4, 16), (5, 35, 8, 1), (600, 97, 8, 16), (70, 30, 16, 13),
                                      (9, 24, 32, 16), (1, 3, 2, 17), (40, 100, 4, 32), (333, 34, 8, 24), (50, 33, 16, 32), (17, 9, 32, 20)])
@pytest.mark.parametrize("lut", ["i8", "f32"])
def test_search_of_few_pairs_up_to_32_centroids(ctx, N, CB, v, C, lut):
    """A wave per token and a few codebooks: indices of the oracle for random rows, near ties on either side of the hysteresis, repeated and
    equal-to-a-centroid rows, NaN and infinities in rows and centroids, padded codebooks, several tokens per wave, both index
    layouts, and rows that are only 4-byte aligned."""
    if kernel_switches():
        pytest.skip("the environment keeps one search for every shape")
    import torch
    M = 20
    x, cent, table, bias = make_case(700 + N + CB, N, CB * v, v, C, M, lut)
    rng = np.random.default_rng(N + C)
    if C > 2:
        cent[::3, C // 2] = cent[::3, 0]                                   # repeated centroids
        cent[1::3, C - 1] = cent[1::3, 1] + np.float32(3e-7)               # ... nearly so: the hysteresis decides
    xv = x.reshape(N, CB, v)
    rows = rng.integers(0, C, (N, CB))
    near = cent[np.arange(CB), rows]                                       # [N][CB][v]
    pick = rng.random((N, CB)) < 0.4
    xv[pick] = near[pick] + rng.choice([0.0, 1e-4, 5e-4], (int(pick.sum()), 1)).astype(np.float32)
    xv[rng.random((N, CB)) < 0.02] = np.nan
    xv[rng.random((N, CB)) < 0.02] = np.inf
    if CB > 4 and C > 1:
        cent[3, rng.integers(0, C)] = np.nan
        cent[4, rng.integers(0, C), 0] = -np.inf
    scales = np.float32(0.0123) if lut == "i8" else None
    want = oracle.index_calculation(x, cent, v, threads=THREADS)
    amm = ctx.amm(cent, table, scales, bias, max_n=N)
    out, idx, _ = amm.run_debug(x, want_acc=False)
    assert np.array_equal(idx, want.reshape(N, CB))
    shifted = torch.empty(N * CB * v + 1, device="cuda")[1:]
    shifted.copy_(torch.from_numpy(x.reshape(-1)).cuda())
    od = torch.empty((N, M), device="cuda")
    torch.cuda.synchronize()
    amm.run_ptr(shifted.data_ptr(), N, od.data_ptr())
    ctx.synchronize()
    assert np.array_equal(od.cpu().numpy().view(np.uint32), out.view(np.uint32))
    amm.close()


@pytest.mark.parametrize("CB,v,C,M", [
    (192, 4, 16, 768),      # column blocks that divide by eight: in order
    (1100, 2, 16, 500),     # 33 column blocks, a table beyond an L2: by XCD
    (1030, 2, 11, 1024),    # 66 of them, padded codebooks
    (400, 2, 16, 333),      # 21, a small table: in order
    (700, 2, 8, 700),       # two codebooks of 8 per entry
    (96, 8, 32, 784), (50, 4, 20, 2304), (60, 4, 64, 1001), (33, 4, 200, 768),   # byte adder
])
def test_items_of_few_tokens(ctx, CB, v, C, M):
    """Launches of one to a few token tiles, in items of 16, 32 and 64 tokens and in order or by XCD, at the edges of each: accumulators and
    output bits of the oracle, nothing behind the output."""
    import torch
    sizes = (1, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 96, 97, 112, 129, 160, 192, 241, 300)
    x, cent, lut, bias = make_case(5200 + CB + M, max(sizes), CB * v, v, C, M)
    want, want_idx, want_acc = oracle.amm_cpu(x, cent, lut, bias, v, 0.0123, 0.0, threads=THREADS)
    amm = ctx.amm(cent, lut, np.float32(0.0123), bias, max_n=max(sizes))
    xd = torch.from_numpy(x).cuda()
    items, guarded = set(), torch.empty((max(sizes) + 3, M), device="cuda")
    for n in sizes:
        out, idx, acc = amm.run_debug(x[:n])
        name = amm.last_gather_kernel()
        assert np.array_equal(idx, want_idx[:n]) and np.array_equal(acc, want_acc[:n]), (n, name)
        assert np.array_equal(out.view(np.uint32), want[:n].view(np.uint32)), (n, name)
        guarded.fill_(-5.0)
        torch.cuda.synchronize()
        amm.run_ptr(xd.data_ptr(), n, guarded.data_ptr())
        ctx.synchronize()
        items.add(amm.last_gather_kernel())
        got = guarded.cpu().numpy()
        assert np.array_equal(got[:n].view(np.uint32), want[:n].view(np.uint32)) and (got[n:] == -5.0).all(), (n, name)
    if ctx.device_info()["compute_units"] == 256 and not kernel_switches():
        few = [k for k in items if "_few_" in k]
        assert len(few) >= 2, items
        if CB > 1000:
            assert any("true" in k for k in few), items
    amm.close()


@pytest.mark.parametrize("N,CB,M,C,width,groups", [(1000, 8, 768, 16, 48, 3), (513, 640, 760, 16, 48, 3), (300, 33, 1000, 16, 64, 2), (200, 70, 1500, 9, 96, 2),
                                                   (449, 12, 1500, 16, 96, 3), (400, 130, 2049, 16, 64, 2), (65, 96, 9001, 16, 48, 0), (64, 40, 9001, 16, 48, 3),
                                                   (20, 40, 9001, 16, 48, 1), (1, 5, 16001, 16, 48, 1), (700, 129, 1100, 13, 96, 3)])
def test_launches_of_few_tokens_with_several_column_groups(ctx, N, CB, M, C, width, groups):
    """Between the launches of few tokens and the large ones: workgroups of two and three column groups, their column blocks dealt to the
    XCDs (those past the last do nothing), waves with and without K-steps, ragged tokens and columns: accumulators and output bits of the oracle,
    nothing behind the output.  `groups`: column groups of a workgroup on 256 CUs (0: the large kernel)."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about the library's choice")
    import torch
    v = 2
    x, cent, lut, bias = make_case(3100 + N + M, N, CB * v, v, C, M)
    want, want_idx, want_acc = oracle.amm_cpu(x, cent, lut, bias, v, 0.0123, 0.0, threads=THREADS)
    amm = ctx.amm(cent, lut, np.float32(0.0123), bias, max_n=N, tuning={"gather_kernel": pimdl.GATHER_SPARSE, "col_block": width})
    out, idx, acc = amm.run_debug(x)
    name = amm.last_gather_kernel()
    if ctx.device_info()["compute_units"] == 256:
        assert name.startswith("gather_sparse_kernel<" if groups == 0 else "gather_sparse_few_kernel<" if groups == 1 else "gather_sparse_few_wide_kernel<"), name
        assert groups < 2 or name.endswith(f", {groups}>"), name
    assert np.array_equal(idx, want_idx) and np.array_equal(acc, want_acc), name
    assert np.array_equal(out.view(np.uint32), want.view(np.uint32)), name
    guarded = torch.full((N + 3, M), -5.0, device="cuda")
    xd = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    amm.run_ptr(xd.data_ptr(), N, guarded.data_ptr())
    ctx.synchronize()
    got = guarded.cpu().numpy()
    assert np.array_equal(got[:N].view(np.uint32), want.view(np.uint32)) and (got[N:] == -5.0).all(), name
    amm.close()


@pytest.mark.parametrize("N,M,tuning", [(16384, 4096, {}), (16640, 4160, {}), (17000, 4001, {}), (34000, 2112, {"col_block": 48}),
                                        (33792, 2048, {"col_block": 64, "xcd_col_split": 2}), (65600, 1030, {"token_item": 128}),
                                        (17408, 4096, {"col_block": 96, "xcd_col_split": pimdl.XCD_PLAIN})])
def test_sparse_gather_of_large_outputs(ctx, N, M, tuning):
    """Outputs from 256 MiB on go through the launch in blocks of token tiles, dealt by XCD or in plain order, the last block smaller:
    every row as in launches of a few thousand tokens, which have no blocks, and nothing behind the output."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about the sparse gather")
    import torch
    assert N * M * 4 >= 256 << 20
    v, CB, C = 4, 8, 16
    _, cent, lut, bias = make_case(515 + M, 1, CB * v, v, C, M)
    x = torch.randn((N, CB * v), device="cuda", generator=torch.Generator(device="cuda").manual_seed(N))
    amm = ctx.amm(cent, lut, np.float32(0.0123), bias, max_n=N, tuning=tuning)
    out = torch.full((N + 2, M), -5.0, device="cuda")
    part = torch.empty((4096, M), device="cuda")
    torch.cuda.synchronize()
    amm.run_ptr(x.data_ptr(), N, out.data_ptr())
    ctx.synchronize()
    assert amm.last_gather_kernel().startswith("gather_sparse_blocks_kernel<"), amm.last_gather_kernel()
    assert bool((out[N:] == -5.0).all())
    for i in range(0, N, 4096):
        n = min(4096, N - i)
        torch.cuda.synchronize()
        amm.run_ptr(x[i:].data_ptr(), n, part.data_ptr())
        ctx.synchronize()
        assert torch.equal(out[i:i + n], part[:n]), i
    n = 300
    want = oracle.amm_cpu(x[:n].cpu().numpy(), cent, lut, bias, v, 0.0123, 0.0, threads=THREADS)[0]
    assert np.array_equal(out[:n].cpu().numpy().view(np.uint32), want.view(np.uint32))
    amm.close()


@pytest.mark.parametrize("N,CB,M,act,tuning,form", [
    (32700, 64, 2060, 0, {"col_block": 48}, "<3, 4, 64, 8>"),               # eight waves by the launch rule
    (17000, 70, 4001, 0, {"col_block": 48, "token_item": 512, "cb_per_slice": 32}, "<3, 4, 32, 8>"),
    (17000, 70, 4001, 0, {"col_block": 64, "token_item": 512}, "<4, 4, 32, 8>"),
    (16500, 40, 4096, 0, {"col_block": 64, "token_item": 512, "cb_per_slice": 16}, "<4, 4, 16, 8>"),
    (18000, 40, 3800, 0, {"col_block": 96, "token_item": 512, "cb_per_slice": 16}, "<6, 4, 16, 8>"),
    (17000, 200, 4000, 1, {"col_block": 96}, "<6, 4, 16, 4>"),              # many slices, GELU
    (16390, 96, 4096, 1, {"col_block": 64}, "<4, 4, 32, 4>"),
    (33000, 33, 2100, 1, {"col_block": 48, "token_item": 128}, "<3, 2, 32, 4>"),
])
def test_forms_of_the_sparse_gather_of_large_outputs(ctx, N, CB, M, act, tuning, form):
    """Four and eight waves, slices of 16, 32 and 64 codebooks, several to an item, with GELU too: every row as in launches without blocks."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about the sparse gather")
    import torch
    assert N * M * 4 >= 256 << 20
    v, C = 2, 16
    _, cent, lut, bias = make_case(717 + M + CB, 1, CB * v, v, C, M)
    x = torch.randn((N, CB * v), device="cuda", generator=torch.Generator(device="cuda").manual_seed(N))
    amm = ctx.amm(cent, lut, np.float32(0.0023), bias, max_n=N, tuning=tuning, activation=pimdl.ACT_GELU_TANH if act else pimdl.ACT_NONE)
    out = torch.full((N + 2, M), -5.0, device="cuda")
    part = torch.empty((4096, M), device="cuda")
    torch.cuda.synchronize()
    amm.run_ptr(x.data_ptr(), N, out.data_ptr())
    ctx.synchronize()
    if ctx.device_info()["compute_units"] == 256:
        assert amm.last_gather_kernel() == "gather_sparse_blocks_kernel" + form
    assert bool((out[N:] == -5.0).all())
    for i in range(0, N, 4096):
        n = min(4096, N - i)
        torch.cuda.synchronize()
        amm.run_ptr(x[i:].data_ptr(), n, part.data_ptr())
        ctx.synchronize()
        assert torch.equal(out[i:i + n], part[:n]), i
    if not act:
        n = 200
        want = oracle.amm_cpu(x[:n].cpu().numpy(), cent, lut, bias, v, 0.0023, 0.0, threads=THREADS)[0]
        assert np.array_equal(out[:n].cpu().numpy().view(np.uint32), want.view(np.uint32))
    amm.close()


@pytest.mark.parametrize("act", [pimdl.ACT_NONE, pimdl.ACT_GELU_TANH])
@pytest.mark.parametrize("N,CB,M", [
    (16500, 16, 260),   # rows of no whole half lines, 16 MiB and more: plain stores
    (16100, 16, 260),   # below: streamed
    (16500, 16, 261), (16500, 16, 262), (16300, 8, 259),  # widths that 16 bytes do not divide, either side of 16 MiB
    (4200, 260, 1028),  # a table of more than 4 MiB: streamed
    (4200, 260, 1027), (4200, 240, 1084),
])
def test_sparse_gather_of_rows_that_end_within_lines(ctx, N, CB, M, act):
    """Both kinds of stores in every tile width, the oracle's bits without an activation and otherwise the same as 4-byte stores give."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about the sparse gather")
    import torch
    v, C = 2, 16
    x, cent, lut, bias = make_case(88 + M + CB, N, CB * v, v, C, M)
    xd = torch.from_numpy(x).cuda()
    want = oracle.amm_cpu(x, cent, lut, bias, v, 0.0123, 0.0, threads=THREADS)[0] if act == pimdl.ACT_NONE else None
    for tuning in ({"col_block": 48}, {"col_block": 64}, {"col_block": 96}, {"col_block": 64, "token_item": 128}, {"col_block": 48, "cb_per_slice": 16}):
        amm = ctx.amm(cent, lut, np.float32(0.0123), bias, max_n=N, activation=act, tuning=dict(tuning, gather_kernel=pimdl.GATHER_SPARSE))
        out = torch.full((N + 2, M), -5.0, device="cuda")
        torch.cuda.synchronize()
        amm.run_ptr(xd.data_ptr(), N, out.data_ptr())
        ctx.synchronize()
        assert amm.last_gather_kernel().startswith("gather_sparse_"), amm.last_gather_kernel()
        if want is None:
            want = amm.run_debug(x)[0]  # (with the sums, which takes every column's store by itself)
        assert bool((out[N:] == -5.0).all())
        assert np.array_equal(out[:N].cpu().numpy().view(np.uint32), want.view(np.uint32)), tuning
        amm.close()


def test_sparse_gather_of_rows_that_end_within_lines_takes_no_longer(ctx):
    """11 codebooks, 1112 columns, 16034 tokens took 2.1 times as long as 1120 columns, whose rows are 35 lines; 17 codebooks, 2890 columns 1.5 times as 2912."""
    for n, cb, ragged, whole in ((16034, 11, 1112, 1120), (8936, 17, 2890, 2912)):
        a, b = (gather_us(ctx, n, cb, 16, m) for m in (ragged, whole))
        assert a < 1.35 * b, (n, cb, ragged, a, b)


@pytest.mark.parametrize("N,CB,M,form", [
    (8300, 97, 1100, "blocks_kernel<4, 4, 16, 4>"),        # three workgroups per CU: just beyond two of them, ragged tokens and columns
    (7700, 128, 1088, "blocks_kernel<4, 4, 16, 4>"),
    (8300, 100, 816, "blocks_kernel<3, 4, 16, 4>"),
    (8192, 128, 1024, "blocks_kernel<4, 4, 32, 4>"),       # exactly two workgroups per CU
    (8300, 96, 1100, "blocks_kernel<4, 4, 32, 4>"),        # a sum of 96 codebooks
    (40000, 130, 104, "kernel<4, 4, 32, 4, false>"),       # below 16 MiB: no blocks
    (65000, 130, 104, "blocks_kernel<4, 4, 32, 4>"),
    (17000, 130, 2001, "blocks_kernel<4, 4, 16, 4>"),      # several rounds, odd columns
])
def test_sparse_gather_with_three_workgroups_per_cu(ctx, N, CB, M, form):
    """Either side of the lines between two and three workgroups per CU and of the blocks of token tiles: every row as in launches of 900
    tokens, which have neither, the oracle's bits in the first and last rows, nothing behind the output."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about the library's choice")
    import torch
    v, C = 2, 16
    _, cent, lut, bias = make_case(2025 + M + CB, 1, CB * v, v, C, M)
    x = torch.randn((N, CB * v), device="cuda", generator=torch.Generator(device="cuda").manual_seed(N))
    width = 16 * int(form.split("<")[1][0])
    amm = ctx.amm(cent, lut, np.float32(0.0123), bias, max_n=N, tuning={"col_block": width})
    out = torch.full((N + 2, M), -5.0, device="cuda")
    part = torch.empty((900, M), device="cuda")
    torch.cuda.synchronize()
    amm.run_ptr(x.data_ptr(), N, out.data_ptr())
    ctx.synchronize()
    if ctx.device_info()["compute_units"] == 256:
        assert amm.last_gather_kernel() == "gather_sparse_" + form, amm.last_gather_kernel()
    assert bool((out[N:] == -5.0).all())
    for i in range(0, N, 900):
        n = min(900, N - i)
        torch.cuda.synchronize()
        amm.run_ptr(x[i:].data_ptr(), n, part.data_ptr())
        ctx.synchronize()
        assert torch.equal(out[i:i + n], part[:n]), i
    rows = list(range(70)) + list(range(N - 70, N))
    want = oracle.amm_cpu(x[rows].cpu().numpy(), cent, lut, bias, v, 0.0123, 0.0, threads=THREADS)[0]
    assert np.array_equal(out[rows].cpu().numpy().view(np.uint32), want.view(np.uint32))
    amm.close()


@pytest.mark.parametrize("N,M,count", [(29200, 768, 3), (22100, 1536, 2), (32768, 1024, 3)])
def test_operators_side_by_side_with_a_large_output(ctx, N, M, count):
    """One gather launch for several operators whose common output is dealt out in blocks: every column as of the operator alone, whose
    output has no blocks."""
    if kernel_switches():
        pytest.skip("a kernel this test is about is switched off by the environment")
    import torch
    assert N * M * count * 4 >= 256 << 20 > N * M * 4
    v, CB, C = 4, 32, 16
    amms = []
    for i in range(count):
        _, cent, lut, bias = make_case(818 + i, 1, CB * v, v, C, M)
        amms.append(ctx.amm(cent, lut, np.float32(0.01 * (i + 1)), bias, max_n=N))
    group = ctx.amm_group(amms)
    assert group.fused_cols == M * count
    x = torch.randn((N, CB * v), device="cuda", generator=torch.Generator(device="cuda").manual_seed(N))
    out = torch.full((N + 1, M * count), -5.0, device="cuda")
    alone = torch.empty((N, M), device="cuda")
    torch.cuda.synchronize()
    group.run_fused_ptr(x.data_ptr(), N, out.data_ptr())
    for i, amm in enumerate(amms):
        amm.run_ptr(x.data_ptr(), N, alone.data_ptr())
        ctx.synchronize()
        assert torch.equal(out[:N, i * M:(i + 1) * M], alone), i
        torch.cuda.synchronize()
    assert bool((out[N:] == -5.0).all())
    group.close()
    for amm in amms:
        amm.close()


@pytest.mark.parametrize("N,CB,C,M", [(16384, 130, 8, 4096), (16384, 160, 3, 4096), (16640, 130, 8, 4160)])
def test_large_outputs_of_up_to_8_centroids(ctx, N, CB, C, M):
    """More than 128 codebooks and 96-column tiles by themselves the best launch: the sparse kernel, also where rows of whole 16 KiB make it
    64-column tiles; the bits of the paired kernel's operator, and of the oracle."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about the library's choice")
    import torch
    v = 2
    _, cent, lut, bias = make_case(615 + M + C, 1, CB * v, v, C, M)
    x = torch.randn((N, CB * v), device="cuda", generator=torch.Generator(device="cuda").manual_seed(N + C))
    outs = [torch.full((N + 2, M), -5.0, device="cuda") for _ in range(2)]
    torch.cuda.synchronize()
    for tuning, out in zip(({}, {"gather_kernel": pimdl.GATHER_ONEHOT}), outs):
        amm = ctx.amm(cent, lut, np.float32(0.0123), bias, max_n=N, tuning=tuning)
        amm.run_ptr(x.data_ptr(), N, out.data_ptr())
        ctx.synchronize()
        name = amm.last_gather_kernel()
        if ctx.device_info()["compute_units"] == 256:
            assert name.startswith("gather_onehot_kernel<" if tuning else "gather_sparse_blocks_kernel<"), name
        amm.close()
    assert torch.equal(outs[0][:N], outs[1][:N]) and bool((outs[0][N:] == -5.0).all())
    n = 200
    want = oracle.amm_cpu(x[:n].cpu().numpy(), cent, lut, bias, v, 0.0123, 0.0, threads=THREADS)[0]
    assert np.array_equal(outs[0][:n].cpu().numpy().view(np.uint32), want.view(np.uint32))


def gather_us(ctx, N, CB, C, M, lut="i8", tuning=None, v=4, group=0):
    """Shortest of a few timings of an operator's gather, us."""
    import torch
    _, cent, table, bias = make_case(1, 1, CB * v, v, C, M, lut)
    scales = None if lut == "f32" else np.full((CB + group - 1) // group, 0.01, np.float32) if group else np.float32(0.01)
    amm = ctx.amm(cent, table, scales, bias, max_n=N, tuning=tuning or {}, scale_group=group)
    x, y = torch.randn(N, CB * v, device="cuda"), torch.empty(N, M, device="cuda")
    torch.cuda.synchronize()
    us = min(amm.profile(x.data_ptr(), N, y.data_ptr(), warmup=8, iters=10)["gather_ms"] for _ in range(5)) * 1e3
    amm.close()
    return us


def test_byte_adder_writes_large_outputs_like_the_sparse_gather(ctx):
    """One codebook: the launch is its stores.  No wait of the epilogue stands between them: 0.94 of the sparse kernel's time, 1.45 with
    the bias of a column chunk loaded behind the stores of the chunk before it.  (Not at every width: rows of 4096 floats, a power of
    two apart, take 1.33, and took 1.58.)"""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about what the caller names")
    rows, sparse = (gather_us(ctx, 38004, 1, 16, 3131, tuning={"gather_kernel": k}) for k in (pimdl.GATHER_ROWS, pimdl.GATHER_SPARSE))
    assert rows < 1.25 * sparse, (rows, sparse)


@pytest.mark.parametrize("M", [99, 258, 1001, 5])
@pytest.mark.parametrize("C", [20, 64, 130])
def test_byte_adder_stores_rows_of_any_width(ctx, C, M):
    """Rows that are no whole float4s, behind an address that is a multiple of 4 bytes only: every bit, and what lies around them."""
    import torch
    N, CB = 700, 40
    x, cent, lut, bias = make_case(9800 + C + M, N, CB * 4, 4, C, M)
    amm = ctx.amm(cent, lut, np.float32(0.02), bias, max_n=N)
    guarded = torch.full((1 + N * M + 64,), -1e30, device="cuda")
    xd = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    amm.run_ptr(xd.data_ptr(), N, guarded.data_ptr() + 4)
    ctx.synchronize()
    assert "gather_i8_" in amm.last_gather_kernel() or kernel_switches(), amm.last_gather_kernel()
    got = guarded.cpu().numpy()
    acc = oracle.gather_i8(oracle.index_calculation(x, cent, 4, threads=THREADS), lut, threads=THREADS)
    want = oracle.dequant(acc, bias, CB, 0.02, 0.0, 0, threads=THREADS)
    assert np.array_equal(got[1:1 + N * M].reshape(N, M).view(np.uint32), want.view(np.uint32))
    assert got[0] == np.float32(-1e30) and (got[1 + N * M:] == np.float32(-1e30)).all()
    amm.close()


def test_odd_widths_of_17_to_32_centroids_are_not_slower_than_the_sparse_gather(ctx):
    """The library gives them to the byte adder: 0.7 of the sparse kernel's time, 1.25 and 1.4 when it stored float by float."""
    if kernel_switches():
        pytest.skip("the environment keeps one kernel for every shape; this test is about the library's choice")
    for N, CB, M in ((20000, 1, 1001), (20000, 33, 258)):
        auto, sparse = (gather_us(ctx, N, CB, 32, M, tuning=t) for t in (None, {"gather_kernel": pimdl.GATHER_SPARSE}))
        assert auto < 1.1 * sparse, (N, CB, M, auto, sparse)


@pytest.mark.parametrize("N,CB,C,M", [(328, 40, 32, 2157), (1500, 33, 16, 905), (1500, 40, 8, 898), (3000, 33, 16, 140),   # column blocks: 135, 57, 57, 9
                                      (2600, 33, 16, 4096), (2600, 3, 32, 4096), (2600, 40, 7, 4095),                  # outputs of 40 MB
                                      (16400, 3, 16, 4096), (32801, 33, 32, 2048)])                                    # of 256 MB, rows of whole 8 KiB
def test_float_tables_whose_column_blocks_do_not_divide_among_the_xcds(ctx, N, CB, C, M):
    """Column blocks dealt out by XCD with some past the last, and in order: every output bit, and the guard rows."""
    import torch
    x, cent, table, bias = make_case(9700 + N + M, N, CB * 4, 4, C, M, "f32")
    amm = ctx.amm(cent, table, None, bias, max_n=N)
    guarded = torch.full((N + 3, M), -1e30, device="cuda")  # no sum of the case comes near it
    xd = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    amm.run_ptr(xd.data_ptr(), N, guarded.data_ptr())
    ctx.synchronize()
    assert "_f32_rows_" in amm.last_gather_kernel(), amm.last_gather_kernel()
    got = guarded.cpu().numpy()
    rows = np.unique(np.concatenate([np.arange(min(N, 70)), np.arange(max(0, N - 70), N), np.arange(250, min(N, 260))]))
    want = oracle.gather_f32(oracle.index_calculation(x[rows], cent, 4, threads=THREADS), table, bias, threads=THREADS)
    assert np.array_equal(got[rows].view(np.uint32), want.view(np.uint32)) and (got[N:] < -9e29).all() and (got[:N] > -9e29).all()
    amm.close()


def test_float_gathers_do_not_depend_on_a_multiple_of_eight_column_blocks(ctx):
    """135 and 136 column blocks of a table beyond the caches, few tokens (2.1 times as long when the 135 were not dealt out by XCD);
    256 and 254 of one codebook, an output beyond the caches (1.5 times when the 256 were)."""
    few = [gather_us(ctx, 328, 192, 32, M, "f32") for M in (2157, 2173)]
    wide = [gather_us(ctx, 6664, 1, 16, M, "f32") for M in (4096, 4064)]   # not 4080: rows just short of 16 KiB take 1.5 times as long in either order
    assert few[0] < 1.4 * few[1], few
    assert wide[0] < 1.3 * wide[1], wide


def test_float_gathers_of_rows_of_up_to_4_kib_are_dealt_out_by_xcd(ctx):
    """32 and 33 column blocks of one codebook, outputs of 180 MB (1.36 times as long when the 32 were taken in order)."""
    a, b = gather_us(ctx, 92160, 1, 16, 512, "f32"), gather_us(ctx, 89367, 1, 16, 528, "f32")
    assert a < 1.2 * b, (a, b)


def test_float_gathers_take_whole_workgroups_where_the_copies_are_the_chain(ctx):
    """32 centroids: 283 tokens in two workgroups per column block, as 400 are (1.5 times their time in five of 64 tokens)."""
    a, b = (gather_us(ctx, n, 768, 32, 3370, "f32", v=1) for n in (283, 400))
    assert a < 1.2 * b, (a, b)


@pytest.mark.parametrize("CB,M,N,kernel", [
    (64, 128, 500, "gather_i8_few_kernel<"), (192, 128, 512, "gather_i8_few_kernel<"), (192, 128, 1024, "gather_i8_few_kernel<"),
    (192, 128, 1040, "gather_i8_kernel<"), (768, 80, 816, "gather_i8_few_kernel<"),     # column blocks that divide by eight, few of them
    (768, 496, 256, "gather_i8_few_kernel<"),                                           # 31 blocks by XCD, two rounds
    (192, 600, 208, "gather_i8_kernel<"),                                               # 38 of them, three rounds of an XCD
    (192, 528, 128, "gather_i8_kernel<"), (384, 265, 250, "gather_i8_kernel<"),         # in order, tables beyond an L2
])
def test_gather_of_64_centroids_by_what_an_xcd_has_to_do(ctx, CB, M, N, kernel):
    """Which of the byte adder's kernels a launch takes, whatever its batch: the rounds of the fullest XCD, and what an XCD reads of the
    table.  Accumulators and output bits of the oracle with either, nothing behind the output."""
    import torch
    v, C = 1, 64
    x, cent, lut, bias = make_case(6700 + M + N, N, CB * v, v, C, M)
    want, _, want_acc = oracle.amm_cpu(x, cent, lut, bias, v, 0.0123, 0.0, threads=THREADS)
    amm = ctx.amm(cent, lut, np.float32(0.0123), bias, max_n=N)
    _, _, acc = amm.run_debug(x)
    assert np.array_equal(acc, want_acc)
    xd, out = torch.from_numpy(x).cuda(), torch.full((N + 2, M), -5.0, device="cuda")
    torch.cuda.synchronize()
    amm.run_ptr(xd.data_ptr(), N, out.data_ptr())
    ctx.synchronize()
    if ctx.device_info()["compute_units"] == 256 and not kernel_switches():
        assert amm.last_gather_kernel().startswith(kernel), amm.last_gather_kernel()
    got = out.cpu().numpy()
    assert np.array_equal(got[:N].view(np.uint32), want.view(np.uint32)) and (got[N:] == -5.0).all()
    amm.close()


@pytest.mark.parametrize("N,CB,C,M,kernel", [
    (17, 48, 64, 3072, "gather_i8_few_kernel<1, 8, false>"),    # rounds that overlap
    (5, 8, 64, 5120, "gather_i8_few_kernel<1, 8, false>"), (25, 11, 200, 6144, "gather_i8_few_kernel<1, 8, false>"),
    (300, 48, 64, 3072, "gather_i8_kernel<"),
    (76, 100, 200, 2048, "gather_i8_few_kernel<1, 8, true>"),   # a table no L2 holds: its token tiles together, also of blocks that eight divides
    (33, 300, 128, 2441, "gather_i8_few_kernel<1, 8, true>"),   # 153 blocks: seven of the grid's past the last
    (40, 20, 64, 1216, "gather_i8_few_kernel<1, 16, false>"), (40, 20, 64, 1200, "gather_i8_few_kernel<1, 16, false>"),  # 76 and 75 blocks
    (17, 512, 24, 8192, "gather_i8_few_kernel<2, 8, false>"),
    (50, 300, 200, 520, "gather_i8_few_kernel<1, 16, true>"),   # 33 blocks, by XCD for the size of the table
    (409, 300, 128, 266, "gather_i8_kernel<"),
])
def test_byte_adder_of_few_tokens_and_many_column_blocks(ctx, N, CB, C, M, kernel):
    """The items that the launch takes by its prices: accumulators and output bits of the oracle, nothing behind the output."""
    import torch
    x, cent, lut, bias = make_case(9100 + M + N, N, CB, 1, C, M)
    want, _, want_acc = oracle.amm_cpu(x, cent, lut, bias, 1, 0.0123, 0.0, threads=THREADS)
    amm = ctx.amm(cent, lut, np.float32(0.0123), bias, max_n=N)
    _, _, acc = amm.run_debug(x)
    assert np.array_equal(acc, want_acc)
    xd, out = torch.from_numpy(x).cuda(), torch.full((N + 2, M), -5.0, device="cuda")
    torch.cuda.synchronize()
    amm.run_ptr(xd.data_ptr(), N, out.data_ptr())
    ctx.synchronize()
    if ctx.device_info()["compute_units"] == 256 and not kernel_switches():
        assert amm.last_gather_kernel().startswith(kernel), amm.last_gather_kernel()
    got = out.cpu().numpy()
    assert np.array_equal(got[:N].view(np.uint32), want.view(np.uint32)) and (got[N:] == -5.0).all()
    amm.close()


def test_byte_adder_of_large_tables_reads_them_once(ctx):
    """76 tokens, five tiles of 16, read 200 MB five times over: 45 us, where 300 tokens on the large kernel take 31 (25 by XCD)."""
    a, b = (gather_us(ctx, n, 256, 200, 3072, v=1) for n in (76, 300))
    assert a < 0.95 * b, (a, b)


@pytest.mark.parametrize("CB,lut,group,M", [(96, "f32", 0, 2441), (768, "f32", 0, 2441), (96, "i8", 8, 3692)])
def test_few_tokens_of_64_centroids_take_the_large_gather_where_it_is_shorter(ctx, CB, lut, group, M):
    """93 tokens, gathered piece by piece, took 1.4 to 1.7 times as long as 150 on the large kernel."""
    a, b = (gather_us(ctx, n, CB, 64, M, lut, v=1, group=group) for n in (93, 150))
    assert a < 1.2 * b, (a, b)


def test_float_gathers_write_rows_of_whole_8_kib_as_fast_as_others(ctx):
    """Outputs of 590 and 440 MB, one codebook (2.9 times as long per byte in workgroups of 256 tokens, column blocks in order)."""
    a, b = (gather_us(ctx, 36000, 1, 16, M, "f32") / M for M in (4096, 3072))
    assert a < 1.5 * b, (a, b)


def test_float_gathers_of_uneven_column_blocks_do_not_wait_for_one_xcd(ctx):
    """38 column blocks on 8 XCDs: 26 token tiles of them took a fifth round of the CUs (1.24 times as long as 24 tiles)."""
    a, b = (gather_us(ctx, n, 96, 8, 608, group=8) for n in (6444, 6144))
    assert a < 1.15 * b, (a, b)


def test_grouped_float_gathers_take_whole_workgroups_from_two_per_cu_on(ctx):
    """8 centroids, a scale per 8 codebooks: 3080 tokens in workgroups of 64 took 1.5 times as long as 3400 in workgroups of 256."""
    a, b = (gather_us(ctx, n, 768, 8, 768, group=8) for n in (3080, 3400))
    assert a < 1.2 * b, (a, b)


def test_byte_adder_writes_whole_rows_of_outputs_beyond_the_caches(ctx):
    """24 centroids, one codebook, 450 MB: 1.2 times the sparse kernel's time when an XCD wrote its own columns of all rows.  (1.07 to 1.10 now, of the
    shortest of eight taken in turn; one against one it is 1.03 .. 1.15.)"""
    rows, sparse = (min(us) for us in zip(*[[gather_us(ctx, 36621, 1, 24, 3072, tuning={"gather_kernel": k}) for k in (pimdl.GATHER_ROWS, pimdl.GATHER_SPARSE)]
                                            for _ in range(8)]))
    assert rows < 1.12 * sparse, (rows, sparse)


@pytest.mark.parametrize("N,C,M", [(20490, 24, 4096), (24570, 64, 3500)])  # 21 token tiles of 1024, and 24, which eight XCDs share
def test_byte_adder_deals_outputs_beyond_the_caches_out_by_tokens(ctx, N, C, M):
    import torch
    x, cent, lut, bias = make_case(9900 + C, N, 12, 4, C, M)
    amm = ctx.amm(cent, lut, np.float32(0.02), bias, max_n=N, tuning={"gather_kernel": pimdl.GATHER_ROWS})
    guarded = torch.full((N + 3, M), -1e30, device="cuda")
    xd = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    amm.run_ptr(xd.data_ptr(), N, guarded.data_ptr())
    ctx.synchronize()
    assert "gather_i8_kernel" in amm.last_gather_kernel(), amm.last_gather_kernel()
    got = guarded.cpu().numpy()
    pick = np.unique(np.concatenate([np.arange(0, N, 97), np.arange(1000, 1050), np.arange(N - 70, N)]))
    acc = oracle.gather_i8(oracle.index_calculation(x[pick], cent, 4, threads=THREADS), lut, threads=THREADS)
    want = oracle.dequant(acc, bias, 3, 0.02, 0.0, 0, threads=THREADS)
    assert np.array_equal(got[pick].view(np.uint32), want.view(np.uint32)) and (got[N:] < -9e29).all() and (got[:N] > -9e29).all()
    amm.close()
