"""Rules of the host side, run without a GPU: which entry points a call goes to, on a library that only notes what is called, and the kernel
library's own plans."""

from __future__ import annotations

import ctypes

import pytest
import torch

from prefixserve_amd.build import ensure_kernels
from prefixserve_amd.kernels.ops import _SIGNATURES, HipOps


class NotingLibrary:
    """Every entry point returns 0 and is noted with its arguments."""

    def __init__(self) -> None:
        self.calls: list[tuple[str, tuple]] = []

    def __getattr__(self, name: str):
        def entry(*args):
            self.calls.append((name, args))
            return 0

        return entry


class Buffers:
    def __init__(self) -> None:
        self.asked: dict[str, int] = {}

    def get(self, name, shape, dtype):
        out = torch.empty(shape, dtype=dtype)
        self.asked[name] = max(self.asked.get(name, 0), out.numel())
        return out


@pytest.fixture
def ops():
    made = object.__new__(HipOps)
    made.device, made.lib, made.ws, made._step_stream = torch.device("cpu"), NotingLibrary(), Buffers(), 0
    made.linear = lambda x, w, out: None                 # the router's logits
    return made


def experts_called(ops, t: int, k: int, f: int, experts: int = 8, top: int = 2) -> list[str]:
    """The entry points of one routed layer, a grouped call marked with whether the router sorted its pairs."""
    x = torch.empty(t, k, dtype=torch.bfloat16)
    router = torch.empty(experts, k)
    chosen, weight = torch.empty(t, top, dtype=torch.int32), torch.empty(t, top)
    ops.moe_route(x, router, chosen, weight, router.to(torch.bfloat16), **({"expert_width": f} if f % 64 else {}))
    w_in, w_down = torch.empty(experts, 2 * f, k, dtype=torch.bfloat16), torch.empty(experts, k, f, dtype=torch.bfloat16)
    ops.moe_experts(x, chosen, weight, w_in, w_down, torch.empty(t * top, f, dtype=torch.bfloat16), torch.empty(top, t, k), 1.0, 7.0, 0.0)
    done = {"psamd_moe_experts_grouped": lambda a: f" sorted {a[18]}"}
    return [name + done.get(name, lambda a: "")(args) for name, args in ops.lib.calls if name != "psamd_moe_grouped_max_tiles"]


PAIR_BY_PAIR = ["psamd_moe_topk", "psamd_moe_experts_rows"]
SORTED_BY_THE_ROUTER = ["psamd_moe_topk_group", "psamd_moe_experts_grouped sorted 1"]


@pytest.mark.parametrize("t,k,f,want", [
    (1, 128, 64, SORTED_BY_THE_ROUTER), (2, 64, 192, SORTED_BY_THE_ROUTER),
    (1, 128, 72, PAIR_BY_PAIR), (2, 64, 1000, PAIR_BY_PAIR), (2, 64, 33, PAIR_BY_PAIR), (2, 72, 64, PAIR_BY_PAIR),
    (3, 64, 72, SORTED_BY_THE_ROUTER), (16, 72, 64, SORTED_BY_THE_ROUTER), (3, 64, 33, PAIR_BY_PAIR), (3, 36, 64, PAIR_BY_PAIR),
    (17, 64, 72, ["psamd_moe_topk", "psamd_moe_experts_grouped sorted 0"]),
])
def test_one_and_two_tokens_are_grouped_where_both_widths_are_whole(ops, t, k, f, want):
    """One and two tokens of experts whose width is no multiple of 64 ran in the slower grouped kernel; and the router sorts a step's
    pairs exactly if the experts take them sorted."""
    assert experts_called(ops, t, k, f) == want


@pytest.mark.parametrize("t,experts,want", [
    (2, 1024, SORTED_BY_THE_ROUTER), (1, 1025, PAIR_BY_PAIR), (2, 4097, PAIR_BY_PAIR),
    (3, 1025, ["psamd_moe_topk", "psamd_moe_experts_grouped sorted 0"]),
])
def test_one_and_two_tokens_among_any_number_of_experts(ops, t, experts, want):
    """The sorting refuses more than 4,096 experts, which one and two tokens did not need it for."""
    assert experts_called(ops, t, 64, 64, experts) == want


@pytest.fixture(scope="module")
def planner():
    made = object.__new__(HipOps)
    made.lib, made._plans = ensure_kernels(), {}
    for name in ("psamd_attention_decode_plan", "psamd_linear_skinny_takes", "psamd_linear_skinny_ksplit", "psamd_linear_tile_plan",
                 "psamd_moe_expert_tile_rows", "psamd_moe_experts_tiled"):
        getattr(made.lib, name).argtypes = _SIGNATURES[name]
    made.lib.psamd_last_error.restype = ctypes.c_char_p
    return made


@pytest.mark.parametrize("requests,hq,hkv,d,runs", [
    (21, 32, 8, 64, 3), (22, 32, 8, 64, 1), (31, 128, 8, 32, 1), (32, 32, 8, 64, 1), (40, 32, 8, 64, 1), (176, 16, 1, 64, 1),
    (22, 136, 8, 64, 2), (31, 256, 8, 64, 2), (32, 256, 8, 64, 1), (176, 17, 1, 64, 2), (255, 64, 1, 64, 2), (256, 64, 1, 64, 1), (90, 48, 2, 64, 2),
    (22, 32, 8, 80, 2), (31, 32, 8, 128, 2), (12, 16, 16, 256, 2), (32, 32, 8, 128, 1), (32, 8, 8, 256, 1), (17, 32, 8, 256, 3),
])
def test_keys_stay_whole_where_the_kernel_of_eight_waves_takes_them(planner, requests, hq, hkv, d, runs):
    """From 176 (request, kv head) pairs on there is one run of all keys, but more than 16 query heads a kv head, which that kernel
    does not take, and heads of more than 64, where the longest of uneven contexts would outlast the others, keep two until there is
    a workgroup for every compute unit."""
    assert planner.decode_plan(requests, 2000, False, hkv, 0, hq, d) == (runs, 128)


@pytest.mark.parametrize("m,n,k,here", [
    (77, 2048, 8192, True), (77, 5120, 14336, True), (128, 5120, 32768, True),                     # few rows
    (66, 5184, 4096, True), (96, 8192, 7296, True), (96, 8192, 14336, True), (128, 7168, 4096, True),   # one round of workgroups
    (72, 8192, 4096, True), (72, 8192, 8192, False), (104, 8192, 16384, False), (72, 8192, 32768, True),  # rows a power of two apart
    (104, 6144, 8192, False), (104, 6144, 14336, False), (104, 6144, 16384, False), (96, 10240, 2048, False),   # a second round
    (72, 6144, 18432, True), (72, 5632, 2880, True), (128, 6144, 13888, True), (104, 10240, 24576, False), (72, 9216, 2880, False), (77, 12288, 4096, False), (77, 16384, 20480, False),
])
def test_slices_of_k_are_taken_where_they_are_one_round(planner, m, n, k, here):
    """Products for the stream of 65 to 128 tokens: any K from 14,336 on was taken, also where the slices begin a second round of workgroups, up to 18%
    slower than the library's product, which ran there before."""
    x, w = torch.empty(m, 64, dtype=torch.bfloat16), torch.empty(64, 64, dtype=torch.bfloat16)   # addresses alone are looked at
    takes = planner._through_lds(x, w, x, m, n, k, "residual") and planner.lib.psamd_linear_skinny_ksplit(m, n, k) > 1
    assert takes == here


@pytest.mark.parametrize("n,k", [(6144, 64), (2048, 64)])
def test_a_step_left_to_the_library_asks_for_the_slices_of_a_shorter_one(ops, n, k):
    """Up to 64 tokens a product for the stream has slices whatever its sizes: where 65 to 128 tokens go to the library, their step asks for the
    slices' room too, so that no buffer grows behind the largest step."""
    ops._direct_library, ops.fixed_kv_len, ops._slice_views, ops._fuses = True, None, {}, {}
    ops.lib.psamd_linear_skinny_takes = lambda *args: 0              # the library's
    ops.lib.psamd_linear_skinny_ksplit = lambda m, n, k: 4
    x, w = torch.empty(100, k, dtype=torch.bfloat16), torch.empty(n, k, dtype=torch.bfloat16)
    large = ops.linear_to_residual(x, w, "o")
    assert large.shape == (100, n) and large.dtype == torch.bfloat16
    asked = dict(ops.ws.asked)
    assert ops.linear_to_residual(x[:40], w, "o").shape == (4, 40, n)
    assert ops.ws.asked == asked


LIBRARY, SLICES, GATED = -1, 0, 2


def plan_of(shape: int, slices: int = 1) -> int:
    return 16 * shape + slices


@pytest.mark.parametrize("m,n,k,silu,gelu", [
    (640, 8192, 2048, plan_of(0), LIBRARY), (1531, 4096, 2048, plan_of(0), LIBRARY), (4096, 8192, 2048, plan_of(0), LIBRARY),   # the library is faster
    (2048, 2816, 1024, plan_of(0), plan_of(1)), (900, 6144, 1024, plan_of(0), plan_of(1)),       # smaller tiles are
    (900, 8192, 3072, plan_of(0), plan_of(0)), (1023, 8192, 2048, plan_of(0), plan_of(0)),       # faster there all the same
    (256, 8192, 2048, plan_of(3), plan_of(3)), (535, 8192, 2048, LIBRARY, LIBRARY),
])
def test_the_largest_tiles_count_what_gelu_takes(planner, m, n, k, silu, gelu):
    """Their activations run with no matrix instruction beside them: GELU takes longer than the SiLU that the table was made for."""
    assert [planner.lib.psamd_linear_tile_plan(GATED, m, n, k, act) for act in (0, 1, 2)] == [silu, silu, gelu]


@pytest.mark.parametrize("m,n,k,want", [
    (516, 6960, 5440, plan_of(1, 3)), (786, 5232, 6656, LIBRARY), (711, 3376, 8320, plan_of(2, 2)),    # 252 tiles, 33 of them on a die of 32 units
    (413, 4992, 7744, plan_of(0, 6)), (422, 3344, 10880, plan_of(0, 8)), (796, 4016, 5696, plan_of(0, 4)),    # one round, up to 256 tiles
])
def test_the_largest_tiles_count_the_rounds_that_are_launched(planner, m, n, k, want):
    """Products for the stream: three and six slices have 80 and 40 workgroups each, a die's eighth of a slice's tiles walked by an eighth of those.
    Where all the tiles together are one round of the chip, a die's may be two."""
    assert planner.lib.psamd_linear_tile_plan(SLICES, m, n, k, 0) == want
    shape, slices = divmod(want, 16)
    if want != LIBRARY and shape == 0:
        tiles = -(-m // 256) * -(-n // 256)
        assert -(-tiles // 8) <= 256 // slices // 8


@pytest.mark.parametrize("m,n,k,want", [
    (262, 6944, 7552, plan_of(2, 2)), (281, 6880, 7168, plan_of(2, 2)), (285, 4496, 15424, plan_of(2, 3)), (253, 4544, 14464, plan_of(3, 3)),   # slower in the largest
    (555, 7552, 5696, LIBRARY), (518, 7792, 6784, LIBRARY),                  # and in two slices of them
    (1009, 2528, 7616, plan_of(0, 4)), (301, 5520, 9280, plan_of(0, 4)),     # close to the library by the table, but faster
    (422, 3344, 10880, plan_of(0, 8)), (1023, 4096, 14336, plan_of(0, 4)),
])
def test_the_largest_tiles_replace_smaller_ones_by_a_lead(planner, m, n, k, want):
    """Products for the stream: where the table has the largest tiles and smaller ones within its own error, the smaller ones stay."""
    assert planner.lib.psamd_linear_tile_plan(SLICES, m, n, k, 0) == want


@pytest.mark.parametrize("tokens,k,f,experts,rows", [
    (24000, 3264, 256, 5, 256), (24000, 3264, 192, 5, 128), (100000, 192, 3264, 8, 128), (16384, 2048, 1024, 32, 256),
    (24000, 256, 72, 5, 0), (512, 2048, 1024, 32, 0),
])
def test_tiles_of_256_pairs_come_with_four_steps_of_k_or_more(planner, tokens, k, f, experts, rows):
    """Their next tile's pairs are asked for behind a tile's first step and used three steps in front of its end: with fewer steps than four the next
    tile's copies would take this one's pairs. Asked for all the same, they are refused on the host."""
    assert planner.lib.psamd_moe_expert_tile_rows(tokens, k, f, experts, 0, 1, 0) == rows
    for short_k, short_f in ((192, 256), (256, 192), (64, 64)):
        assert planner.lib.psamd_moe_experts_tiled(*[None] * 8, 1, 100, short_k, short_f, 2, 0, 1, 1.0, 7.0, 0.0, 1, 0, 0, None, 256) == 1
        assert b"too few steps" in planner.lib.psamd_last_error()
