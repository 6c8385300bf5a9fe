"""The rules by which kernels are chosen, asked on the host: no GPU is needed to ask."""
import pytest
import torch

from tessweave_engine_amd.kernels import ops
from tessweave_engine_amd.kernels.lib import library

F32, BF16 = 0, 1


@pytest.mark.parametrize("m,n,k,ranges", [(489, 5496, 4736, 2), (1900, 3584, 18944, 2), (536, 5120, 13824, 4)])
def test_products_that_one_kernel_does_not_take_keep_the_plan_of_the_other(m, n, k, ranges):
    """Four columns more than a multiple of 8: results are not rows of 16 bytes, so that the tiles whose waves take turns do not run,
    and the K ranges are those of the tiles that do. The scratch holds either plan's."""
    lib = library()
    assert lib.tw_linear_partial_splits_rows(BF16, 1, m, n + 4, k, k) == ranges
    assert lib.tw_linear_workspace_bytes(BF16, m, n + 4, k) >= ranges * m * (n + 4) * 4
    for cols in (n, n + 4):
        named = lib.tw_linear_partial_splits_rows(BF16, 1, m, cols, k, k)
        assert lib.tw_linear_workspace_bytes(BF16, m, cols, k) >= named * m * cols * 4


@pytest.mark.parametrize("dtype,m,n,k,whole", [(BF16, 8, 2048, 2304, True), (BF16, 8, 2304, 2560, False), (BF16, 8, 2304, 2816, True), (BF16, 1, 2304, 3584, False),
                                               (BF16, 8, 2560, 3584, True), (BF16, 9, 2560, 3584, False), (F32, 8, 2560, 1536, False), (F32, 8, 2560, 1792, True),
                                               (F32, 1, 2560, 2304, False), (F32, 8, 3072, 2816, True), (F32, 8, 3072, 3328, False), (F32, 8, 3584, 3584, True),
                                               (F32, 8, 3584, 3328, False), (F32, 9, 3584, 2048, False)])
def test_sums_for_the_next_kernel_over_the_whole_of_k(dtype, m, n, k, whole):
    """Up to 8 rows and a long K: K ranges stay where they are the faster form, one workgroup a CU of whole stages."""
    assert (library().tw_linear_partial_splits_rows(dtype, 1, m, n, k, k) == 1) == whole


@pytest.mark.parametrize("dtype,n,k,here,apart", [(BF16, 7168, 5120, (), (3, 6, 10, 16)), (BF16, 10240, 5120, (), (1, 3, 6, 16)), (BF16, 10240, 3584, (), (1, 6, 16)),
                                                  (BF16, 4608, 8192, (), (1, 6, 16)), (F32, 5120, 3072, (), (1, 3, 16)), (F32, 4608, 3584, (), (1, 6)),
                                                  (BF16, 4096, 5120, (1, 6, 10), (16,)), (BF16, 9216, 2048, (1, 3, 6), (16,)), (BF16, 7168, 4096, (1, 3, 6), ()),
                                                  (BF16, 1152, 896, (1, 8, 16), ()), (F32, 7168, 2048, (1, 3, 6), ()), (BF16, 7168, 3072, (1, 3, 6), (16,))])
def test_products_that_rotate_where_they_are_faster(dtype, n, k, here, apart):
    """Measured beside split sums that another kernel finishes; those kept apart are 1 to 40 % slower in one (and so are some near the line)."""
    pays = library().tw_linear_rotate_pays
    assert all(pays(dtype, m, n, k) for m in here) and not any(pays(dtype, m, n, k) for m in apart)


@pytest.mark.parametrize("rows", [1, 8])
def test_an_activation_behind_few_rows_asks_for_what_its_kernel_takes(rows):
    """Rows 2,050 elements apart are no multiple of 16 bytes apart, which the kernel refuses of a single row too."""
    weight = ops.shuffle_weight(torch.zeros(4096, 2048, dtype=torch.bfloat16))
    assert ops.linear_act_few_pays(torch.zeros(rows, 2048, dtype=torch.bfloat16), weight)
    assert ops.linear_act_few_pays(torch.zeros(rows + 1, 2056, dtype=torch.bfloat16)[:rows, :2048], weight)
    assert not ops.linear_act_few_pays(torch.zeros(rows + 1, 2050, dtype=torch.bfloat16)[:rows, :2048], weight)


@pytest.mark.parametrize("dtype,heads,kv_heads,dim,value_dim,n,keys,good", [
    ("bfloat16", 16, 4, 128, 128, 1, 320, {5}), ("bfloat16", 16, 4, 128, 128, 16, 48, {1}), ("bfloat16", 1, 1, 128, 128, 2, 68, {1}),
    ("bfloat16", 24, 4, 128, 128, 200, 100, {1}), ("float32", 16, 4, 128, 128, 1, 128, {4}), ("bfloat16", 30, 10, 64, 64, 93, 645, {5, 11}),
    ("bfloat16", 20, 10, 128, 128, 64, 600, {4}), ("float32", 20, 10, 128, 128, 1, 80, {5}), ("bfloat16", 16, 4, 128, 256, 130, 400, {4, 5}),
    ("float32", 24, 12, 128, 128, 24, 700, {9, 10}), ("bfloat16", 16, 4, 192, 128, 4, 3000, set(range(47, 65)))])
def test_key_ranges_of_mixed_heads_fill_whole_rounds(dtype, heads, kv_heads, dim, value_dim, n, keys, good):
    """Where the ranges measured beside one another lie 3 % apart and more: the fastest, for the kernel whose waves have a key head each and
    for the other."""
    kind = getattr(torch, dtype)
    k, v = torch.empty(1, kv_heads, 16, dim, dtype=kind), torch.empty(1, kv_heads, value_dim, 16, dtype=kind)
    assert ops.attn_mixed_splits(n, keys, heads, k, v) in good


@pytest.mark.parametrize("dtype,heads,kv_heads,dim,n,good", [
    ("bfloat16", 28, 4, 128, 5, {768: {8, 9, 10, 11, 12}, 6144: {11, 12}, 12288: {11, 12}, 32768: {12}}), ("bfloat16", 28, 4, 128, 7, {6144: {8, 9}, 12288: {8, 9}, 32768: {9}}),
    ("bfloat16", 28, 4, 128, 8, {3072: {8}, 6144: {8}, 12288: {8, 16}, 32768: {8, 16}}), ("bfloat16", 28, 4, 128, 9, {3072: {7}, 6144: {7, 14}, 12288: {7}, 32768: {7}}),
    ("bfloat16", 28, 4, 128, 12, {3072: {5}, 12288: {5}}), ("bfloat16", 28, 4, 128, 16, {1500: {4}, 3072: {4, 8}, 12288: {4, 8}}),
    ("bfloat16", 28, 4, 128, 32, {768: {2, 3, 4}, 3072: {2}, 6144: {2}}), ("bfloat16", 14, 2, 64, 16, {3072: {8}, 12288: {8}}),
    ("float32", 28, 4, 128, 8, {3072: {8}, 12288: {8}}), ("float32", 28, 4, 128, 4, {768: {12, 14, 16}, 12288: {16}}), ("float32", 14, 2, 64, 24, {3072: {5}, 12288: {5}})])
def test_key_ranges_of_one_token_sequences_fill_whole_turns(dtype, heads, kv_heads, dim, n, good):
    """The ranges measured within some 3 % of the fastest; a full turn and part of another is up to a quarter behind. And a captured step's
    workspace holds what any length class up to the cache's asks for."""
    kind = getattr(torch, dtype)
    for keys, ranges in good.items():
        assert ops.attn_decode_splits(n, heads, kv_heads, keys, dim, kind) in ranges, keys
    for bound in (1 << i for i in range(4, 16)):
        for span in (0, 100, 4096):
            splits, most = ops.attn_decode_class_splits(n, heads, kv_heads, bound, 32768, span, dim, kind)
            assert 1 <= splits <= most <= 64


@pytest.mark.parametrize("bound,keys,want", [(0, 30000, 44), (32768, 30000, 44), (4096, 3000, 16)])
def test_key_ranges_of_a_context_made_by_hand(monkeypatch, bound, keys, want):
    """A context without a length class asks for its longest sequence's ranges."""
    from types import SimpleNamespace
    from tessweave_engine_amd.parts.attention import paged_attention
    seen = []
    monkeypatch.setattr(ops, "attn_decode", lambda *a, **k: seen.append(k["splits"]))
    ctx = SimpleNamespace(n_decode=1, n_seqs=1, n_tokens=1, capturing=False, kv_bound=bound, max_kv_len=keys, kv_capacity=32768, q_start=None, kv_len=None,
                          workspace=SimpleNamespace(get=lambda tag, shape, dtype: torch.empty(shape, dtype=dtype)))
    paged_attention(ctx, torch.empty(1, 28 * 128, dtype=torch.bfloat16), None, None, SimpleNamespace(block_table=None), None, 28, 4, 128, 0.1)
    assert abs(seen[0] - want) <= 3


def test_key_ranges_are_estimated_once_for_the_layers_of_a_step(monkeypatch):
    shape = (13, 28, 4, 2048, 8192, 0, 128, torch.bfloat16)
    want = ops.attn_decode_class_splits(*shape)
    monkeypatch.setattr(ops, "library", lambda: pytest.fail("estimated again"))
    assert ops.attn_decode_class_splits(*shape) == want


@pytest.mark.parametrize("heads,kv_heads,dim,value_dim,page", [(16, 4, 128, 128, 16), (1, 1, 64, 64, 32), (20, 10, 128, 128, 16), (16, 4, 128, 128, 24)])
def test_no_length_has_more_key_ranges_than_a_workspace_is_sized_for(heads, kv_heads, dim, value_dim, page):
    """A captured step's workspace is sized once for all lengths up to the cache's."""
    k, v = torch.empty(1, kv_heads, page, dim), torch.empty(1, kv_heads, value_dim, page)
    for n in (1, 3, 16, 100, 1024, 2000):
        most = [ops.attn_mixed_most_splits(n, length) for length in (1, 100, 1000, 8000)]
        assert most == sorted(most) and most[-1] <= 64
        assert all(1 <= ops.attn_mixed_splits(n, length, heads, k, v) <= most[-1] for length in range(1, 8000, 37))


@pytest.mark.parametrize("latent,rotated,heads,n,length,good", [(192, 64, 16, 28, 1092, {6, 7, 8, 9}), (128, 64, 32, 10, 1590, set(range(9, 13))), (192, 64, 16, 8, 190, {3}),
                                                                (192, 64, 16, 1, 2050, {33}), (192, 64, 24, 9, 1733, {14}), (128, 64, 16, 174, 1149, {1}),
                                                                (240, 16, 32, 92, 633, {2}), (112, 48, 16, 175, 1142, {2}), (240, 16, 16, 21, 4764, set(range(19, 25)))])
def test_key_ranges_of_a_cached_latent_fill_whole_rounds(latent, rotated, heads, n, length, good):
    """Where the ranges measured beside one another lie 3 % apart and more: the fastest. And no length has more than a workspace is sized for."""
    keys, values = torch.empty(1, 1, 16, latent + rotated), torch.empty(1, 1, latent, 16)
    assert ops.latent_decode_splits(n, heads, length, keys, values) in good
    most = ops.latent_decode_most_splits(n, heads, length)
    assert most <= 64 and all(1 <= ops.latent_decode_splits(n, heads, t, keys, values) <= most for t in range(1, length, 13))


@pytest.mark.parametrize("window,keep_first", [(1024, 0), (1024, 8), (50, 0)])
def test_key_ranges_of_a_window_hold_the_tiles_that_it_touches(monkeypatch, window, keep_first):
    """A window that ends inside a tile touches one tile more than a window of whole tiles: no range of the step has a fifth."""
    from types import SimpleNamespace
    from tessweave_engine_amd.parts.windowed import mixed_attention
    seen = []
    monkeypatch.setattr(ops, "attn_mixed", lambda *a, **k: seen.append(k["splits"]))
    keys = torch.empty(1, 4, 16, 128)
    ctx = SimpleNamespace(n_decode=1, n_seqs=1, capturing=False, kv_bound=4096, max_kv_len=4000, kv_capacity=4096, q_start=None, kv_len=None,
                          workspace=SimpleNamespace(get=lambda tag, shape, dtype: torch.empty(shape, dtype=dtype)))
    mixed_attention(ctx, None, keys, torch.empty(1, 4, 128, 16), SimpleNamespace(block_table=None), None, 16, 4, 128, 0.1, window=window,
                    keep_first=keep_first)
    tiles = max(len({j // 16 for j in range(p - window + 1, p + 1)} | {j // 16 for j in range(keep_first)}) for p in range(3900, 3950))
    assert -(-tiles // seen[0]) <= 4
