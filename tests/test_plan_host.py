"""What the plan of multi-token products decides, on the CPU: it is a function of shapes, token counts and the CU count (256 before a
device has set it), so no device is needed.  Reached through the library's own C++ symbols."""
import ctypes as C

import pytest

import cases as K
import oracle as O
import whole_rows as W

QUANTIZED = [K.Q4_0, K.Q5_0, K.Q5_1, K.Q8_0, K.Q4_K, K.Q6_K]


@pytest.fixture(scope="module")
def act_workspace(lib):
    f = getattr(lib, "_ZN2nh24gemm_act_workspace_bytesEPKNS_7MatViewEjjbb")
    f.restype, f.argtypes = C.c_size_t, [C.POINTER(W.MatView), C.c_uint32, C.c_uint32, C.c_bool, C.c_bool]

    def workspace(ty, rows, cols, tokens, epilogue):
        return f(W.views(ty, rows, cols), len(rows), tokens, epilogue, False)
    return workspace


@pytest.fixture(scope="module")
def whole_rows(lib):
    return lambda *product: W.planned(lib, *product)


@pytest.mark.parametrize("ty", QUANTIZED, ids=lambda t: O.TYPE_NAMES[t])
def test_variants_are_what_the_gpu_tests_take_them_for(whole_rows, ty):
    for rows, cols, tokens, wg_rows, waves in W.VARIANTS[ty] + W.CHAINED[ty]:
        assert whole_rows(ty, [rows], cols, tokens) == (wg_rows, waves), (rows, cols, tokens)


@pytest.mark.parametrize("ty", QUANTIZED, ids=lambda t: O.TYPE_NAMES[t])
def test_a_product_that_writes_over_its_input_shares_columns(whole_rows, ty):
    """A workgroup that owns whole rows stores them while others still read x.  With shared columns and more than 32 tokens x is cut by a
    launch of its own before any result is stored."""
    n, x = 1024, 1 << 32
    size = 4 * 64 * n
    apart = whole_rows(ty, [n], n, 64, [x], [x + size])
    assert apart[0] in (16, 32, 64) and apart == whole_rows(ty, [n], n, 64)
    assert apart == whole_rows(ty, [n], n, 64, [x], [x - size])
    for y in (x, x + 4, x + size - 4, x - size + 4):
        assert whole_rows(ty, [n], n, 64, [x], [y]) == (0, 0)
    # another product's input, in one launch
    assert whole_rows(ty, [n, n], n, 64, [x, x + size], [x + 2 * size, x + 3 * size])[0] != 0
    assert whole_rows(ty, [n, n], n, 64, [x, x + size], [x + 2 * size, x]) == (0, 0)


@pytest.mark.parametrize("ty", QUANTIZED, ids=lambda t: O.TYPE_NAMES[t])
def test_an_epilogue_asks_for_all_planned_shares(act_workspace, ty):
    """A chain's product asks for the workspace of its planned column shares whether or not it then takes whole rows, as the same
    product without an epilogue does; a job whose columns are not shared needs one share for the epilogue to read."""
    for rows, cols in (([4096], 4096), ([512], 512), ([1024], 14336), ([2048, 2048], 2048), ([14336, 14336], 4096), ([32000], 1024)):
        for tokens in (3, 8, 9, 16, 17, 32, 33, 160):
            plain, with_epilogue = act_workspace(ty, rows, cols, tokens, False), act_workspace(ty, rows, cols, tokens, True)
            one = sum((tokens * r * 4 + 255) // 256 * 256 for r in rows)
            assert with_epilogue == max(plain, one), (rows, cols, tokens)


@pytest.mark.parametrize("ty", QUANTIZED, ids=lambda t: O.TYPE_NAMES[t])
def test_cut_activations_start_on_lines(lib, ty):
    """The planes of up to 32 tokens' cut activations (16 bytes a slot) are whole 128-byte lines apart; the slots of the last tile, 16, 32
    or 64, are there, and a buffer made for so many tokens holds them."""
    stride = getattr(lib, "_ZN2nh15act_slot_strideEjj")
    stride.restype, stride.argtypes = C.c_uint32, [C.c_uint32, C.c_uint32]
    for tokens in list(range(3, 130)) + [512, 1000]:
        s = stride(ty, tokens)
        tile = 16 if tokens <= (8 if ty == K.Q6_K else 16) else 32 if tokens <= 32 else 64
        assert s >= (tokens + tile - 1) // tile * tile and s <= tokens + 64
        assert tokens > 32 or s % 8 == 0, tokens


# (dtype, rows, cols, tokens): many rounds of workgroups, measured slower with whole rows by 6 to 33 %
MANY_ROUNDS = [(K.Q4_K, [20000], 256, 9), (K.Q4_K, [20000], 256, 16), (K.Q4_K, [32000], 512, 9), (K.Q4_K, [32000], 512, 16),
               (K.Q4_K, [4096] * 8, 512, 16), (K.Q8_0, [128256], 1024, 16), (K.Q8_0, [64000], 512, 8), (K.Q8_0, [64000], 1024, 8),
               (K.Q4_0, [128256], 256, 8), (K.Q4_0, [128256], 512, 8), (K.Q5_0, [128256], 256, 8)]


@pytest.mark.parametrize("ty,rows,cols,tokens", MANY_ROUNDS, ids=lambda v: str(v))
def test_many_rounds_of_workgroups_share_columns(whole_rows, ty, rows, cols, tokens):
    assert whole_rows(ty, rows, cols, tokens) == (0, 0)


@pytest.mark.parametrize("ty,rows,cols,tokens,want", [
    (K.Q4_0, 14336, 4096, 8, 64), (K.Q4_0, 4096, 4096, 8, 16), (K.Q4_K, 16384, 1024, 12, 32), (K.Q4_K, 12288, 1024, 16, 32),
    (K.Q8_0, 32000, 1024, 8, 64), (K.Q4_0, 512, 2048, 40, 16)], ids=lambda v: str(v))
def test_few_rounds_take_whole_rows(whole_rows, ty, rows, cols, tokens, want):
    assert whole_rows(ty, [rows], cols, tokens)[0] == want


# (dtype, rows, cols, tokens): [gate,up] pairs that lost 8 to 28 % with the launch behind them
LONG_PAIRS = [(K.Q4_0, 14336, 4096, 9), (K.Q4_0, 14336, 8192, 16), (K.Q5_0, 14336, 4096, 16), (K.Q5_0, 14336, 8192, 3), (K.Q4_K, 14336, 512, 9),
              (K.Q4_K, 11008, 1024, 16), (K.Q8_0, 8192, 2048, 33), (K.Q8_0, 8192, 2048, 32), (K.Q4_K, 4096, 1024, 17), (K.Q5_0, 2048, 2048, 160)]


@pytest.mark.parametrize("ty,rows,cols,tokens", LONG_PAIRS, ids=lambda v: str(v))
def test_long_pairs_share_columns(whole_rows, ty, rows, cols, tokens):
    """In a chain the launch that would sum the shares runs in either case: a long pair gains nothing by whole rows."""
    assert whole_rows(ty, [rows, rows], cols, tokens) == (0, 0)


@pytest.mark.parametrize("ty,rows,cols,tokens", [(K.Q4_0, 2816, 1024, 8), (K.Q8_0, 4096, 1024, 16), (K.Q4_K, 2048, 512, 24), (K.Q5_0, 1024, 1024, 100)],
                         ids=lambda v: str(v))
def test_short_pairs_take_whole_rows(whole_rows, ty, rows, cols, tokens):
    assert whole_rows(ty, [rows, rows], cols, tokens)[0] != 0


@pytest.mark.parametrize("ty,rows,cols,tokens", [(K.Q8_0, 4096, 8192, 8), (K.Q4_K, 4096, 8192, 8), (K.Q6_K, 1024, 4096, 3), (K.Q6_K, 2048, 4096, 8),
                                                 (K.Q6_K, 8192, 4096, 8)], ids=lambda v: str(v))
def test_products_a_chain_loses_more_on_than_one_alone_gains(whole_rows, ty, rows, cols, tokens):
    assert whole_rows(ty, [rows], cols, tokens) == (0, 0)


@pytest.mark.parametrize("ty,rows,cols,tokens", [(K.Q4_0, 12288, 11264, 6), (K.Q5_0, 24576, 5120, 4), (K.Q5_0, 24576, 3072, 72), (K.Q8_0, 17408, 3072, 72)],
                         ids=lambda v: str(v))
def test_long_products_share_columns(whole_rows, ty, rows, cols, tokens):
    """Measured slower with whole rows by 12 to 27 %: what a launch less gains does not pay for the activations' cutting there."""
    assert whole_rows(ty, [rows], cols, tokens) == (0, 0)
