"""The library's own rules at sizes on both sides of their lines, on 256 compute units (which it assumes where there is no GPU): which kernel
makes a product of a prompt's rows, and which contexts the 32-bit attention shares out."""
from types import SimpleNamespace

import pytest
import torch

from geneinfer_amd.kernels import ops
from geneinfer_amd.parts.linear import linear, linear_onto

# m, n, k, what becomes of the sums -> the kernel that was the faster one there, by more than 4 %
MEASURED = [
    (2600, 4096, 128, "stored", "128x128"), (2600, 4096, 512, "stored", "128x128"), (2048, 4096, 768, "stored", "128x128"), (1777, 5120, 3072, "stored", "256x128"),
    (1300, 6144, 256, "stored", "128x128"), (2048, 3072, 2048, "stored", "256x128"),
    (2048, 3072, 512, "added", "256x128"), (2048, 3072, 2048, "added", "256x128"), (2600, 2048, 256, "added", "256x128"), (3000, 3072, 8192, "added", "256x128"),
    (3000, 3072, 256, "added handing a norm on", "128x128"), (2600, 4096, 256, "added handing a norm on", "128x128"), (2048, 3072, 2048, "added handing a norm on", "256x128"),
    (3000, 3072, 8192, "added handing a norm on", "256x128"),
    (3000, 3072, 256, "rotated", "128x128"), (2048, 5120, 1024, "rotated", "128x128"), (1777, 6144, 1024, "rotated", "128x128"), (2048, 3072, 2048, "rotated", "256x128"),
    (777, 5120, 3072, "rotated", "256x128"),
    (300, 16384, 2048, "gated", "256x128"), (256, 16384, 2048, "gated", "128x128"), (2048, 16384, 2048, "gated", "256x256"), (1500, 16384, 2048, "gated with a norm", "256x256"),
    (8192, 28672, 4096, "gated with a norm", "256x256"), (1777, 8192, 2048, "xielu", "256x256"), (2048, 2048, 2048, "added", "128x128"), (300, 2048, 2048, "added", "128x128 shared"),
    (128, 4096, 4096, "stored", None), (200, 4096, 100, "stored", None),
]


@pytest.mark.parametrize("m,n,k,kind,kernel", MEASURED)
def test_the_faster_kernel_is_chosen(m, n, k, kind, kernel):
    assert ops.gemm_bf16_large_kernel(m, n, k, kind) == kernel


@pytest.mark.parametrize("m,n,k,kernel", [(129, 16384, 2048, "strips"), (192, 16384, 3072, "strips"), (193, 16384, 2048, "128x128"), (131, 28672, 4096, "256x128"), (131, 16384, 2056, None),
                                          (184, 12288, 2048, "strips"), (160, 12288, 3072, "strips"), (184, 12288, 3072, "128x128"), (160, 12288, 4096, "strips"), (160, 12288, 6144, "256x128"),
                                          (150, 13056, 14336, "256x128"), (192, 16384, 4096, "strips"), (192, 16384, 6144, "256x128")])
def test_strips_where_one_round_of_them_is_faster(m, n, k, kernel):
    assert ops.gemm_bf16_large_kernel(m, n, k, "gated") == kernel


# m, n, k, gated -> the kernel of up to 128 rows that was the faster one there, by more than 4 % or (on one side of a line) as fast
FEW_ROWS = [
    (1, 12288, 2048, True, "slim"), (8, 12288, 2048, True, "slim"), (10, 12288, 2048, True, "strips"), (12, 12288, 1024, True, "slim"), (16, 12288, 1024, True, "strips"), (1, 16384, 3072, True, "slim"),
    (16, 16384, 2048, True, "slim"), (16, 18432, 4096, True, "slim"), (8, 28672, 4096, True, "slim"), (10, 28672, 4096, True, "slim"), (12, 28672, 4096, True, "strips"), (16, 36864, 3072, True, "slim"),
    (8, 12288, 256, True, "slim"), (16, 20480, 512, True, "slim"), (1, 33280, 64, True, "strips"), (8, 28672, 384, True, "slim"), (9, 28672, 384, True, "strips"),
    (1, 12288, 3072, False, "slim"), (8, 12288, 2048, False, "slim"), (12, 12288, 2048, False, "strips"), (12, 13824, 1024, False, "slim"), (16, 13824, 1024, False, "strips"), (16, 16384, 2048, False, "slim"),
    (16, 20480, 4096, False, "slim"), (16, 28672, 4096, False, "slim"), (12, 28672, 1024, False, "slim"), (16, 28672, 1024, False, "strips"), (16, 33280, 3072, False, "slim"), (5, 128256, 2048, False, "slim"),
    (16, 128256, 2048, False, "slim"), (1, 152064, 64, False, "strips"), (8, 100352, 256, False, "strips"), (8, 65536, 512, False, "slim"), (9, 65536, 512, False, "strips"), (16, 24576, 512, False, "slim"),
    (4, 32000, 384, False, "slim"), (9, 32000, 384, False, "strips"), (4, 28672, 512, False, "slim"), (8, 28672, 512, False, "streamed"), (10, 14336, 512, False, "slim"), (14, 14336, 512, False, "streamed"),
    (20, 16384, 512, False, "strips"), (11, 16384, 2056, True, "slim"), (12, 16384, 2056, True, "streamed"), (16, 3072, 2048, False, "slim"), (17, 3072, 2048, False, "slim tiles"), (17, 3072, 2048, True, "strips"),
    (128, 3072, 2048, False, "strips"), (128, 3072, 2056, False, "streamed"), (129, 3072, 2048, False, None),
]


@pytest.mark.parametrize("m,n,k,gated,kernel", FEW_ROWS)
def test_the_faster_kernel_is_chosen_for_few_rows(m, n, k, gated, kernel):
    assert ops.gemm_bf16_small_kernel(m, n, k, gated) == kernel


# rows, columns, k, distances between rows of either operand in pieces of 16 bytes (None: k), gated, added onto -> weight rows a workgroup, whether it reckons in 64 bits
@pytest.mark.parametrize("m,n,k,lda8,ldw8,gated,added,reach", [
    (16, 8192, 4096, None, None, False, False, (32, False)), (16, 8192, 4096, ((1 << 28) - 512) // 15, None, False, False, (32, False)), (16, 8192, 4096, ((1 << 28) - 512) // 15 + 1, None, False, False, (24, False)),
    (16, 8192, 4096, (1 << 28) // 15, None, False, False, (24, False)), (9, 8192, 4096, ((1 << 28) - 512) // 8, None, False, False, (32, False)), (1, 8192, 4096, 1 << 40, None, False, False, (32, False)),
    (16, 8192, 4096, ((1 << 32) - 512) // 15, None, False, False, (24, False)), (16, 8192, 4096, ((1 << 32) - 512) // 15 + 1, None, False, False, (24, True)), (2, 8192, 4096, 1 << 33, None, False, False, (24, True)),
    (16, 16384, 4096, ((1 << 28) - 512) // 15, None, True, False, (32, False)), (16, 16384, 4096, ((1 << 28) - 512) // 15 + 1, None, True, False, (16, False)), (8, 16384, 4096, (1 << 32) // 7, None, True, False, (16, True)),
    (4, 8192, 4096, None, ((1 << 28) - 512) // 31, False, False, (32, False)), (4, 8192, 4096, None, ((1 << 28) - 512) // 31 + 1, False, False, (24, False)),
    (1, 2, 4096, None, (1 << 32) - 512, False, False, (8, False)), (1, 2, 4096, None, (1 << 32) - 511, False, False, (8, True)), (3, 1, 4096, None, 1 << 40, False, False, (8, False)),
    (8, 4096, 4096, (1 << 32) // 7, None, False, True, (16, True)), (8, 4096, 4096, ((1 << 32) - 512) // 7, None, False, True, (16, False))])
def test_few_rows_far_apart_are_reached(m, n, k, lda8, ldw8, gated, added, reach):
    """The place of a row's last piece holds in the 32 bits that the kernel adds in, bytes or pieces; beyond them nothing is refused, and a sum of squares handed on has as many pieces as ever."""
    lda8, ldw8 = lda8 or k // 8, ldw8 or k // 8
    assert ops.gemm_bf16_slim_reach(m, n, k, 8 * lda8, 8 * ldw8, gated, added) == reach
    rows, far = reach
    last = max((m - 1) * lda8, (7 if gated else min(rows, n) - 1) * ldw8) + k // 8 - 1
    assert far or last * (16 if rows > 24 else 1) < 1 << 32
    if added:
        assert -(-n // rows) == ops.lib().gi_gemm_bf16_norm_parts(m, n, k)


# rows, columns, k, added onto, gated -> weight rows a workgroup: what covers the compute units evenly, in whole groups of 8 where that costs less, few enough for a reader of a norm's pieces
@pytest.mark.parametrize("m,n,k,added,gated,rows", [(1, 2048, 8192, True, False, 8), (8, 2304, 768, False, False, 9), (1, 4096, 4096, True, False, 16), (8, 6144, 4096, False, False, 24), (8, 8192, 512, True, False, 16),
                                                    (16, 8192, 8192, True, False, 16), (1, 8192, 2048, False, False, 32), (8, 12288, 8192, False, False, 24), (8, 128256, 2048, False, False, 32), (8, 16384, 2048, False, True, 32),
                                                    (1, 28672, 4096, False, True, 16), (12, 28672, 4096, False, True, 32)])
def test_weight_rows_of_a_workgroup(m, n, k, added, gated, rows):
    assert ops.gemm_bf16_slim_reach(m, n, k, k, k, gated, added) == (rows, False)


# m, n, k -> tiles of rows and shares of k in strips, or None where the other kernels were the faster ones
@pytest.mark.parametrize("m,n,k,cut", [(131, 3072, 8192, (1, 5)), (256, 3072, 8192, (1, 5)), (301, 2048, 2048, (4, 2)), (300, 3072, 8192, (5, 2)), (300, 3072, 20480, None), (300, 6144, 14336, None),
                                       (131, 10240, 2048, (3, 1)), (131, 10240, 6144, None), (129, 11264, 768, (1, 1)), (256, 11264, 768, None), (400, 500, 4096, (7, 4)), (900, 500, 8192, None),
                                       (256, 500, 8192, (4, 8)), (1400, 320, 28672, None), (1536, 1920, 640, (8, 1)), (1537, 1920, 640, None), (64, 2048, 2048, (1, 4)), (64, 2048, 2056, None),
                                       (64, 16384, 2048, None), (2048, 2048, 2048, None)])
def test_products_are_cut_into_strips_where_that_is_faster(m, n, k, cut):
    assert ops.gemm_bf16_strip_cut(m, n, k) == cut


def test_a_cut_does_not_depend_on_what_was_asked_before():
    """Answers are kept by size: asked in other orders, between others whose answers lie in the same places, and from another thread they are the same."""
    from concurrent.futures import ThreadPoolExecutor
    sizes = [(m, n, k) for m in (17, 49, 131, 163, 300, 332, 1400) for n in (500, 2048, 3072) for k in (512, 2048, 8192)]
    ask = lambda order: {size: ops.lib().gi_gemm_bf16_strip_cut(*size) for size in order}
    first = ask(sizes)
    assert len(set(first.values())) > 10 and ask(sizes[::-1]) == first and ask(sizes[::5] + sizes) == first
    with ThreadPoolExecutor(2) as pool:
        assert all(got == first for got in pool.map(ask, [sizes, sizes[::-1]]))


# m, n, k -> the most shares of k that either kernel makes, as the scratch shows them
@pytest.mark.parametrize("m,n,k,shares", [(131, 3072, 8192, 5), (40, 5120, 3072, 4), (131, 10240, 2048, 2), (256, 3072, 8192, 5), (300, 2048, 2048, 4), (600, 3072, 8192, 2), (17, 200, 64, 1), (40, 128, 12288, 32)])
def test_scratch_holds_as_many_shares_as_either_kernel_makes(m, n, k, shares):
    assert ops._scratch_floats(m, n, k, 0, False) == shares * m * n


# m, n, k, what becomes of the sums, the kernel that was the faster one, by how many workgroups it makes its last tiles, and without counters
SHARED_OR_NOT = [
    (4096, 3072, 8192, "added", "256x256", 1, 1), (4096, 3072, 8192, "stored in bfloat16", "256x256", 1, 1), (1368, 8192, 6784, "stored in bfloat16", "256x256", 1, 1),
    (573, 16384, 6464, "added", "256x256", 1, 1), (709, 16384, 10176, "gated", "256x256", 1, 1), (1161, 8192, 2048, "added", "256x128", 1, 1), (588, 14336, 2048, "added", "256x128", 1, 1),
    (273, 8192, 3072, "added handing a norm on", "128x128", 1, 1), (489, 6144, 3072, "added handing a norm on", "128x128", 1, 1), (793, 2048, 2496, "stored in bfloat16", "128x128", 1, 1),
    (740, 4096, 4096, "added handing a norm on", "256x128", 2, 1), (206, 10240, 2624, "stored in bfloat16", "128x128", 1, 1), (496, 6144, 3136, "rotated", "128x128", 1, 1),
    (318, 512, 4416, "added handing a norm on", "256x128", 4, 4), (437, 8192, 7168, "added handing a norm on", "256x128", 2, 2),
    (2048, 2048, 8192, "added", "256x128", 2, 2), (1777, 2048, 8192, "added handing a norm on", "256x128", 2, 2), (2048, 5120, 3072, "rotated", "256x128", 4, 4),
    (3000, 3072, 8192, "stored", "256x128", 4, 4), (2600, 4064, 4160, "gated", "256x128", 2, 2), (2048, 2048, 2048, "added", "128x128", 1, 1), (2048, 3072, 2048, "xielu", "256x128", 1, 1),
]


@pytest.mark.parametrize("m,n,k,kind,kernel,shares,without", SHARED_OR_NOT)
def test_tiles_are_shared_out_where_that_is_faster(m, n, k, kind, kernel, shares, without):
    number = ops.PRODUCT_KINDS.index(kind)
    assert ops.gemm_bf16_large_kernel(m, n, k, kind) == kernel
    assert (ops._shares(m, n, k, number, True), ops._shares(m, n, k, number, False)) == (shares, without)


def test_only_a_product_whose_tiles_are_shared_out_asks_for_their_scratch():
    """Counters, and 128 KB a share: at most one for every compute unit, so 33.6 MB."""
    asked = 0
    for m in (129, 300, 777, 1000, 1500, 2048, 3000, 4096, 8192):
        for n in (512, 2048, 3072, 5120, 8192, 16384):
            for k in (512, 2048, 3136, 8192):
                for number in range(len(ops.PRODUCT_KINDS)):
                    if ops.gemm_bf16_large_kernel(m, n, k, ops.PRODUCT_KINDS[number]) == "128x128 shared":
                        continue
                    for counted in (True, False):
                        floats, shares = ops._scratch_floats(m, n, k, number, counted), ops._shares(m, n, k, number, counted)
                        assert floats == 0 if shares == 1 else 2 * 32768 <= floats <= 256 * 32768 + 512
                        asked += shares > 1
    assert asked > 100


@pytest.mark.parametrize("rows,seen,spans", [(1, 256, 0), (1, 257, 3), (3, 4096, 17), (1, 65534 * 256, 65535), (1, 65534 * 256 + 1, 0), (1, 1 << 30, 0)])
def test_a_context_is_shared_out_over_so_many_spans_as_a_grid_takes(rows, seen, spans):
    """One head of 16 channels, whose parts are small: longer contexts stay whole (0), they are not refused."""
    assert ops.lib().gi_attention_exact_spans(rows, rows, 1, 1, 16, 16, 16, seen) == spans


# rows, rows of their own, heads, key heads, channels, positions seen -> whether a span's blocks go out one by one; beside it what was measured, microseconds of spans and of blocks
@pytest.mark.parametrize("rows,single,heads,kv,hd,seen,blocks", [(3, 3, 24, 8, 128, 600, True),                                                   # 25.7, 12.9
                                                                 (24, 0, 24, 8, 128, 1000, True), (32, 0, 24, 8, 128, 1000, False), (60, 0, 24, 8, 128, 1000, True),          # 25.5, 20.8; 25.7, 28.4; 46.0, 36.3
                                                                 (100, 0, 16, 16, 128, 300, True), (128, 0, 16, 2, 128, 500, False),               # 26.4, 19.3; 27.8, 30.5
                                                                 (1, 1, 24, 8, 128, 8000, False), (5, 5, 24, 8, 128, 8000, True), (3, 3, 8, 1, 128, 40000, False),              # 37.2, 44.2; 134, 106; 105, 144
                                                                 (10, 10, 8, 1, 128, 12000, False), (14, 14, 8, 1, 128, 12000, True),              # 70.1, 74.1; 91.5, 86.1
                                                                 (12, 12, 32, 8, 64, 600, True), (12, 12, 32, 8, 64, 1000, False), (16, 0, 32, 8, 64, 1000, True), (16, 0, 32, 8, 64, 2000, False),
                                                                 (1, 1, 32, 8, 64, 4000, True), (1, 1, 16, 2, 64, 8000, False)])                   # 20.8, 19.7; 26.9, 28.8
def test_blocks_of_keys_go_out_one_by_one_where_that_is_faster(rows, single, heads, kv, hd, seen, blocks):
    spans, floats = ops._exact_spans(rows, single, heads, kv, hd, hd, 16, -(-seen // 256) * 256)
    assert spans > 1 and floats == rows * heads * spans * (hd + 4) * (4 if blocks else 1)


@pytest.mark.parametrize("m,n,k,taken", [(3, 16384, 2048, 1), (1, 4096, 4096, 1), (8, 8192, 4096, 1), (1, 6656, 4096, 1), (16, 1024, 4096, 1), (1, 1024, 1024, 1), (1, 2048, 2048, 1), (8, 5120, 2048, 1),
                                         (9, 1000, 4096, 1), (1, 1000, 4096, 0), (1, 1024, 4096, 0), (8, 2048, 3072, 0), (1, 5632, 4096, 0), (4, 4608, 3072, 0), (8, 1024, 2048, 0), (2, 6144, 2048, 0), (17, 4096, 1024, 0), (3, 4095, 1024, 0)])
def test_gates_in_the_product_where_that_is_faster(m, n, k, taken):
    assert ops.gemm_exact_gated_pays(m, n, k) == taken


# workgroups uncut, longest context, mean, channels -> cuts, as measured faster
@pytest.mark.parametrize("groups,longest,mean,hd,splits", [(192, 3000, 1640, 128, 2), (168, 2988, 2247, 128, 1), (144, 1709, 1282, 128, 1), (152, 4064, 3041, 64, 1), (176, 6694, 3350, 64, 3), (148, 3501, 1400, 64, 4),
                                                           (128, 1123, 645, 128, 1), (224, 4589, 2300, 128, 2), (64, 500, 100, 128, 1)])
def test_known_contexts_are_cut_where_that_is_faster(groups, longest, mean, hd, splits):
    assert ops._decode_ragged_split(groups, longest, mean, hd, 8) == ((splits, 4) if splits > 1 else (1, 8))


# (first position, rows) of every portion, heads, channels, window -> shares, as measured faster
WALKS = [
    ([(0, 1500)], 32, 64, 0, 3), ([(0, 1024)], 32, 64, 0, 3), ([(0, 800)], 32, 64, 0, 3), ([(2000, 600)], 32, 64, 0, 3), ([(1300, 300), (0, 200)], 32, 64, 0, 3), ([(0, 1777)], 32, 64, 1024, 3),
    ([(0, 1000)] * 2, 32, 64, 0, 1), ([(839, 479)], 64, 64, 0, 1), ([(866, 254)] * 4, 64, 64, 1024, 1), ([(0, 2048)], 32, 64, 1024, 1), ([(0, 950)] * 2, 32, 64, 512, 1), ([(522, 1961)], 32, 64, 0, 1),
    ([(0, 760)], 32, 64, 0, 1), ([(347, 409), (0, 1638), (133, 157), (0, 171), (0, 289), (0, 701)], 32, 64, 1024, 1), ([(0, 2581)], 32, 64, 0, 2),
    ([(0, 1000)], 32, 128, 0, 2), ([(0, 2000)], 24, 128, 0, 2), ([(1000, 1350), (0, 674)], 24, 128, 0, 3), ([(0, 1024)] * 2, 24, 128, 0, 1), ([(0, 2972)], 12, 128, 1024, 1), ([(0, 2048)], 32, 128, 0, 1),
    ([(0, 800)], 32, 128, 0, 1), ([(3000, 700), (0, 700)], 32, 128, 0, 4),
]


def _plan(portions):
    starts = [sum(n for _, n in portions[:i]) for i in range(len(portions))]
    return ops.AttentionPlan(starts, [n for _, n in portions], [p for p, _ in portions], list(range(len(portions))), "cpu")


@pytest.mark.parametrize("portions,heads,hd,window,shares", WALKS)
def test_walks_over_keys_are_shared_out_where_that_is_faster(portions, heads, hd, window, shares):
    plan = _plan(portions)
    one_round = (plan.n_tiles // 2 if plan.paired else plan.n_tiles) * heads <= 256
    assert ops._walk_shares(plan, heads, hd, window, 0, one_round)[0] == shares
    assert list(plan.walk_shares.values())[0][0] == shares


@pytest.mark.parametrize("portions,bracket,heads,hd,shares", [([(0, 1000)], 1024, 32, 64, 3), ([(0, 1000)], 1024, 32, 128, 1), ([(839, 479)], 2048, 64, 64, 1), ([(900, 600)], 2048, 32, 64, 3)])
def test_walks_of_a_captured_pass_go_by_its_bracket(portions, bracket, heads, hd, shares):
    """Whatever the positions of the step it was captured with."""
    found = set()
    for back in (0, 100):
        plan = _plan([(max(0, p - back), n) for p, n in portions])
        plan.max_tile_context, plan.tile_contexts = bracket, None
        found.add(ops._walk_shares(plan, heads, hd, 0, 0, True))
    assert len(found) == 1 and found.pop()[0] == shares


def test_no_room_for_scratch_is_no_error(monkeypatch):
    def full(*args, **kw):
        raise torch.OutOfMemoryError("full")

    assert ops._room(5, "cpu").shape == (5,)
    monkeypatch.setattr(torch, "empty", full)
    assert ops._room(5, "cpu") is None


def _launches_with_room_for(floats, monkeypatch):
    """What is launched from here on, on a device with room for allocations of up to so many numbers."""
    launched, empty = [], torch.empty

    def bounded(*size, **kw):
        if torch.Size(size[0] if len(size) == 1 and not isinstance(size[0], int) else size).numel() > floats:
            raise torch.OutOfMemoryError("full")
        return empty(*size, **kw)

    monkeypatch.setattr(ops, "_dev", lambda *tensors: None)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_call", lambda name, *a: launched.append((name, a)))
    monkeypatch.setattr(torch, "empty", bounded)
    return launched


@pytest.mark.parametrize("rows,hd,seen", [(3, 128, 600), (12, 64, 600)])
def test_attention_without_room_for_blocks_of_keys_goes_by_spans(rows, hd, seen, monkeypatch):
    """The blocks of keys leave four times the numbers that the spans leave: a step that fits with spans is not refused."""
    spans, floats = ops._exact_spans(rows, rows, 24, 8, hd, hd, 16, -(-seen // 256) * 256)
    least = rows * 24 * spans * (hd + 4)
    assert floats == 4 * least
    q, at, cache = torch.zeros(rows, 24 * hd), torch.zeros(rows, dtype=torch.int32), torch.zeros(4, 8 * 16 * 2 * hd)
    out, table = torch.zeros_like(q), torch.zeros(rows, 4, dtype=torch.int32)
    for room, given in ((floats, floats), (floats - 1, least), (least, least)):
        with monkeypatch.context() as patch:
            launched = _launches_with_room_for(room, patch)
            ops.attention_exact(q, cache, out, at, at, table, 24, 8, hd, page_size=16, single_rows=True, max_context=seen)
            assert [(name, a[-3:-1]) for name, a in launched] == [("gi_attention_exact", (given, spans))]


@pytest.mark.parametrize("m,n,k,before", [(33, 3072, 8192, 4), (131, 3072, 8192, 4), (96, 10240, 8192, 2), (40, 128, 12288, 32), (64, 2048, 2056, 8)])
def test_a_product_without_room_for_strips_shares_of_k_has_those_of_before(m, n, k, before, monkeypatch):
    """A step that fits with the sums of the kernels beside strips is not refused, whichever way its product is asked for."""
    wanted, least = ops._scratch_floats(m, n, k, 0, False), before * m * n
    assert wanted >= least and (wanted > least) == ((m, n, k) in [(33, 3072, 8192), (131, 3072, 8192), (96, 10240, 8192)])
    bf16 = lambda *shape: torch.zeros(shape, dtype=torch.bfloat16)
    a, w, x, normed, at = bf16(m, k), bf16(n, k), torch.zeros(m, n), bf16(m, n), torch.zeros(m, dtype=torch.int32)
    cache, table, turns = bf16(2, 2, 8, 64, 64), torch.zeros(1, 2, dtype=torch.int32), torch.zeros(m, 32)
    calls = [(ops.gemm_bf16, (a, w, x))]
    if ops.gemm_bf16_onto_norm_takes(m, n, k):
        calls.append((ops.gemm_bf16_onto_norm, (a, w, x, torch.zeros(n), 1e-6, normed)))
    if n == 3072:
        calls.append((ops.gemm_bf16_qkv_rope_store, (a, w, turns, turns, at, at, table, bf16(m, 32 * 64), cache, 32, 8, 64)))
    for call, args in calls:
        for room, given in ((wanted, wanted), (wanted - 1, least if wanted > least else None), (least, least)):
            if given is None:
                continue
            with monkeypatch.context() as patch:
                launched = _launches_with_room_for(room, patch)
                call(*args)
            (name, passed), = launched
            assert given in passed and (wanted == given or wanted not in passed), name


def test_products_of_few_rows_ask_for_nothing_by_kind(monkeypatch):
    for m, n, k in [(1, 3072, 2048), (17, 2048, 8192), (128, 16384, 2048), (128, 28672, 4096)]:
        assert m <= ops.FEW_ROWS and len({ops._scratch_floats(m, n, k, kind, counted) for kind in range(len(ops.PRODUCT_KINDS)) for counted in (False, True)}) == 1
        assert all(ops._shares(m, n, k, kind, True) == 1 for kind in range(len(ops.PRODUCT_KINDS)))
    asked = []
    for name in ("product_kind", "_shares"):
        monkeypatch.setattr(ops, name, lambda *a, _inner=getattr(ops, name), _name=name, **k: (asked.append(_name), _inner(*a, **k))[1])
    monkeypatch.setattr(ops, "_dev", lambda *tensors: None)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_call", lambda *a: None)
    step = SimpleNamespace(memo={}, device="cpu")
    bf16 = lambda *shape: torch.zeros(shape, dtype=torch.bfloat16)
    for m in (1, 128):
        linear(bf16(m, 2048), bf16(3072, 2048), torch.zeros(m, 3072), ctx=step)
        linear_onto(bf16(m, 2048), bf16(2048, 2048), torch.zeros(m, 2048), None, step)
    assert not asked and not step.memo
    linear(bf16(2048, 8192), bf16(2048, 8192), torch.zeros(2048, 2048), accumulate=True, ctx=step)
    assert asked and step.memo["product_counters"].numel() >= ops.lib().gi_gemm_bf16_counters()


def test_how_a_step_s_attention_is_cut_is_found_once_for_its_layers(monkeypatch):
    asked = []
    for name in ("_decode_ragged_split", "prompt_attention_splits"):
        monkeypatch.setattr(ops, name, lambda *a, _inner=getattr(ops, name), _name=name, **k: (asked.append(_name), _inner(*a, **k))[1])
    launched = []
    monkeypatch.setattr(ops, "_dev", lambda *tensors: None)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_call", lambda name, *a: launched.append((name, a)))
    n_single, heads, n_kv, hd, page = 24, 24, 8, 128, 16
    lens, befores = [1] * n_single + [900], [400 + 110 * i for i in range(n_single)] + [64]
    starts = list(range(n_single)) + [n_single]
    plan = ops.AttentionPlan(starts, lens, befores, list(range(n_single + 1)), "cpu")
    n = sum(lens)
    q = torch.zeros(n, heads * hd, dtype=torch.bfloat16)
    cache, table = torch.zeros(8, 2, n_kv, page, hd, dtype=torch.bfloat16), torch.zeros(n_single + 1, 256, dtype=torch.int32)
    at = torch.zeros(n, dtype=torch.int32)
    memo = {}
    layer = lambda window: ops.attention_bf16(q, cache, torch.zeros_like(q), plan, at, at, table, heads, n_kv, hd, window=window, memo=memo)
    for _ in range(3):
        layer(None)
    assert sorted(asked) == ["_decode_ragged_split", "prompt_attention_splits"]
    layer(512)                                   # (another kind of layer: its own cut)
    assert asked.count("prompt_attention_splits") == 2
    plan.decode_positions = None                 # (a step still to come: nothing that was found of this one holds)
    layer(None)
    splits = [args[-10] for name, args in launched if name == "gi_attention_decode_bf16"]
    assert splits[0] == splits[1] == splits[2] > 1 and splits[-1] == 1


# portions (positions before, rows), single rows at, heads, key heads, channels, window -> workgroups for each single row's context beside the tiles (0: a launch of their own)
@pytest.mark.parametrize("portions,singles,heads,kv,hd,window,splits", [([(1000, 1350), (0, 674)], [380, 3000] * 12, 24, 8, 128, 0, 1), ([(0, 1039)], [1117, 2198], 24, 8, 128, 0, 2),
                                                                        ([(1030, 198), (0, 99)], [2322], 24, 8, 128, 0, 2), ([(0, 607)], [8452], 24, 8, 128, 0, 9),
                                                                        ([(2073, 670), (0, 334)], [5761], 32, 8, 64, 0, 2), ([(0, 300)], [30000] * 30, 24, 8, 128, 0, 0),
                                                                        ([(0, 1000)], [500], 24, 8, 96, 0, 0), ([(0, 300)], [500], 32, 8, 64, 0, 0),
                                                                        # windows: tiles far behind walk no longer than those at the start, and rows far behind read no more than the window
                                                                        ([(60000, 300)], [4096], 8, 2, 128, 4096, 3), ([(4096, 300)], [4096], 8, 2, 128, 4096, 3), ([(0, 300)], [30000] * 30, 24, 8, 128, 512, 1)])
def test_single_rows_beside_tiles(portions, singles, heads, kv, hd, window, splits):
    segs = [(c - 1, 1) for c in singles] + portions
    plan = ops.AttentionPlan([sum(n for _, n in segs[:i]) for i in range(len(segs))], [n for _, n in segs], [p for p, _ in segs], list(range(len(segs))), "cpu")
    seen = lambda context, slack: min(context, window + slack) if window else context
    cut = lambda: (lambda tiles: ops._both_cut(plan, heads, kv, hd, window, 0, 16, seen, tiles[0], tiles[2]))(ops._prompt_cut(plan, heads, hd, window, 0, seen, True))
    assert cut() == splits and cut() == splits
    plan.decode_positions = None                 # a step still to come
    assert cut() == 0


@pytest.mark.parametrize("rows,apart", [([1, 1, 1], True), ([1, 3], False), ([64], False), ([1, 65], True), ([1, 40, 40], True), ([1, 30, 30, 500], False), ([500, 900], True)])
def test_short_portions_go_row_by_row_over_pages_in_common(rows, apart, monkeypatch):
    """What the kernel is told, of itself and where the step says that requests may share pages; a captured step of single rows is told by its step."""
    launched = []
    monkeypatch.setattr(ops, "_dev", lambda *tensors: None)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_call", lambda name, *a: launched.append((name, a)))
    plan, n = _plan([(700, r) for r in rows]), sum(rows)
    q, at = torch.zeros(n, 8 * 64, dtype=torch.bfloat16), torch.zeros(n, dtype=torch.int32)
    cache, table = torch.zeros(4, 2, 2, 16, 64, dtype=torch.bfloat16), torch.zeros(len(rows), 128, dtype=torch.int32)
    assert plan.rows_apart == apart and ops.AttentionPlan.all_decode(3, 1000, "cpu").rows_apart
    for in_common in (False, True):
        ops.attention_bf16(q, cache, torch.zeros_like(q), plan, at, at, table, 8, 2, 64, memo={}, in_common=in_common)
    told = [a[15:17] for name, a in launched if name == "gi_attention_decode_bf16"]
    assert told == ([(n, 1 - apart), (n, 1)] if plan.n_decode else [])


@pytest.mark.parametrize("rule", ["_latent_fold_takes", "decode_attention_shape"])
def test_answers_kept_for_a_step_s_sizes_are_bounded(rule):
    """Rows and contexts change from step to step: a process that runs for long keeps no answer for each."""
    assert getattr(ops, rule).cache_parameters()["maxsize"]
