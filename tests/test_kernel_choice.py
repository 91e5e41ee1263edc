"""The rules that deal the expert products to kernels, asked on the CPU for a device of 256 compute units.

What the GPU tests say about the kernels they exercise is checked here without a GPU, and that between them they
exercise every kernel, so that a change of a rule cannot take a kernel's last test away unseen.  The tiles within a
kernel are held to one another's bits, each of them, and some of each product's to the oracle.
"""

from __future__ import annotations

import subprocess

import pytest

import test_gpu_f32_gemm as f32
import test_gpu_joint_products as joint
import test_gpu_middle_batch_beside as beside
import test_gpu_ragged_widths as ragged
import test_gpu_row_bits as row_bits
import test_gpu_tall_tiles as tall
import test_gpu_tile_choice as tiles
import test_gpu_tile_shapes as shapes
from kernel_choice import (DOWN, GATE_UP, MI355X_CUS, chosen, f32_backward_kernel, forward_kernels, gradient_kernels,
                           joint_kernels, joint_tiles, product_tiles, shared_beside, tiles as product_tile)
from research_amd import build

GATE_UP_KERNELS = {"stream_16x128", "stream_16x64", "stream_32x64", "rows64", "rows64_tail", "half", "half_tail", "rows256",
                   "rows256_tail", "rows256_short", "rows256_short_tail"}
DOWN_KERNELS = {"stream_16x128", "stream_16x64", "stream_32x64", "rows64", "half", "half_deep", "rows256", "rows256_tail"}
GRADIENT_KERNELS = {"half", "half_deep", "rows256", "rows256_tail"}


@pytest.mark.parametrize("tokens,hidden,experts,top_k,inter,forward,gradients", tiles.GROUPED + ragged.SHAPES)
def test_grouped_shapes_take_the_kernels_they_name(tokens, hidden, experts, top_k, inter, forward, gradients):
    assert " ".join(forward_kernels(tokens * top_k, hidden, inter, experts, MI355X_CUS)) == forward
    assert " ".join(gradient_kernels(tokens * top_k, hidden, inter, experts, MI355X_CUS)) == gradients


@pytest.mark.parametrize("tokens,hidden,inter,forward,gradients", tiles.DENSE)
def test_dense_shapes_take_the_kernels_they_name(tokens, hidden, inter, forward, gradients):
    assert " ".join(forward_kernels(tokens, hidden, inter, cus=MI355X_CUS)) == forward
    assert " ".join(gradient_kernels(tokens, hidden, inter, cus=MI355X_CUS)) == gradients


@pytest.mark.parametrize("tokens,hidden,inter,experts,kernels", ragged.LAST_ROWS)
def test_last_row_shapes_take_the_kernels_they_name(tokens, hidden, inter, experts, kernels):
    assert " ".join(forward_kernels(tokens, hidden, inter, experts, MI355X_CUS)) == kernels


def test_every_kernel_is_checked_against_the_oracle():
    forward = [case[5].split() for case in tiles.GROUPED + ragged.SHAPES] + [case[3].split() for case in tiles.DENSE]
    gradients = [case[6].split() for case in tiles.GROUPED + ragged.SHAPES] + [case[4].split() for case in tiles.DENSE]
    assert {gate_up for gate_up, _ in forward} == GATE_UP_KERNELS
    assert {down for _, down in forward} == DOWN_KERNELS
    assert {dz for dz, _ in gradients} == GRADIENT_KERNELS
    assert {dx for _, dx in gradients} == GRADIENT_KERNELS


def test_every_kernel_is_held_to_the_bits_of_the_others():
    seen = set()
    for hidden, inter in row_bits.WIDTHS:
        for rows in row_bits.DENSE_ROWS:
            seen.update(zip((GATE_UP, DOWN), forward_kernels(rows, hidden, inter, cus=MI355X_CUS)))
        for experts in row_bits.EXPERTS:
            for rows in (*row_bits.GROUP_ROWS, row_bits.MOST_ROWS // experts):
                seen.update(zip((GATE_UP, DOWN), forward_kernels(rows * experts, hidden, inter, experts, MI355X_CUS)))
    assert {kernel for product, kernel in seen if product == GATE_UP} >= GATE_UP_KERNELS - {"rows256_short"}
    assert {kernel for product, kernel in seen if product == DOWN} >= DOWN_KERNELS


JOINT_KERNELS = ({"separate", "half", "half_tail", "rows256", "rows256_tail"}, {"separate", "half", "rows256", "rows256_tail"},
                 {"separate", "half_deep", "rows256", "rows256_tail"}, {"separate", "half_deep", "rows256", "rows256_tail"})


@pytest.mark.parametrize("tokens,hidden,experts,top_k,inter,shared,kernels", joint.SHAPES)
def test_joint_shapes_take_the_kernels_they_name(tokens, hidden, experts, top_k, inter, shared, kernels):
    assert " ".join(joint_kernels(tokens, top_k, hidden, inter, shared, experts, MI355X_CUS)) == kernels


@pytest.mark.parametrize("tokens,top_k,hidden,inter,shared,experts,dz,dx", [
    # a few rows per group: a tile each, and how many groups have a row is chance.  Jointly where the rounds hold
    # whatever happens, apart where a few groups more start another round
    (12, 8, 2048, 1408, 2816, 64, "separate", "rows256"),
    (16, 8, 2048, 1408, 2816, 64, "separate", "separate"),
    (24, 8, 2048, 1408, 2816, 64, "separate", "separate"),
    (27, 8, 2048, 1408, 2816, 64, "separate", "separate"),
    (6, 8, 2048, 1408, 2816, 64, "rows256", "separate"),
    (8, 8, 2048, 1408, 2816, 64, "separate", "separate"),
    (21, 3, 1000, 2664, 2664, 24, "separate", "half_deep"),
])
def test_joint_gradients_of_a_few_rows_leave_room_for_more_groups(tokens, top_k, hidden, inter, shared, experts, dz, dx):
    assert joint_kernels(tokens, top_k, hidden, inter, shared, experts, MI355X_CUS)[2:] == [dz, dx]


@pytest.mark.parametrize("reduction,gate_up,down", [(192, "separate", "separate"), (200, "separate", "separate"),
                                                    (224, "separate", "separate"), (232, "half_tail", "half")])
def test_joint_half_tiles_have_the_steps_their_pipeline_wants(reduction, gate_up, down):
    """The shortest reductions in half tiles run in four 32-deep stages, which want eight steps, of either product."""
    assert joint_kernels(1000, 2, reduction, 512, 512, 8, MI355X_CUS)[0] == gate_up
    for inter, shared in ((reduction, reduction), (reduction, 512), (512, reduction)):
        assert joint_kernels(1000, 2, 512, inter, shared, 8, MI355X_CUS)[1] == down


def test_every_joint_kernel_is_held_to_separate_launches():
    for product, names in enumerate(zip(*(case[6].split() for case in joint.SHAPES))):
        assert set(names) == JOINT_KERNELS[product]


@pytest.mark.parametrize("tokens,hidden,experts,inter,launches,larger", f32.BACKWARD_SHAPES)
def test_f32_backward_shapes_take_the_launches_they_name(tokens, hidden, experts, inter, launches, larger):
    assert f32_backward_kernel(tokens, hidden, inter, experts, MI355X_CUS) == launches
    assert f32_backward_kernel(larger[0], hidden, inter, larger[1], MI355X_CUS) == "separate"


def test_joint_launches_deal_every_tile_once():
    binary = build.cache_dir() / build.NATIVE_TEST_NAME
    assert binary.exists(), "run __graft_entry__.build() first"
    proc = subprocess.run([binary.as_posix(), "deal"], capture_output=True, text=True, timeout=110)
    assert proc.returncode == 0 and proc.stdout.strip().endswith("PASS"), proc.stdout + proc.stderr


def test_sizes_out_of_range_have_no_kernel():
    assert chosen(GATE_UP, 0, 64, 64, 1, MI355X_CUS) == chosen(4, 1, 64, 64, 1, MI355X_CUS) == ""
    assert chosen(GATE_UP, 1, 63, 64, 1, MI355X_CUS) == chosen(DOWN, 1, 64, 12, 1, MI355X_CUS) == "general"


@pytest.mark.parametrize("tokens,hidden,experts,top_k,d_ff,shared_width,gate_up,down", beside.SHAPES + [beside.RAGGED])
def test_middle_batches_run_beside_the_launches_they_name(tokens, hidden, experts, top_k, d_ff, shared_width, gate_up, down):
    assert shared_beside(tokens, top_k, hidden, d_ff, shared_width, experts) == [gate_up, down]


@pytest.mark.parametrize("hidden,gate_up", [(2**19 - 128, "router 64x64"), (2**19, "")])
def test_layers_that_copy_their_rows_leave_shared_products_alone(hidden, gate_up):
    """x of 1 GiB or more: the routed products read a copy, and the shared ones run behind them."""
    assert shared_beside(1024, 2, hidden, 1984, 576, 16)[0] == gate_up


def test_every_launch_and_tile_beside_it_is_checked():
    launches = [f"{launch} {tile}" for launch in ("router", "dispatch") for tile in ("64x64", "128x64")]
    assert {case[6] for case in beside.SHAPES} == {"", *launches}
    assert {case[7] for case in beside.SHAPES} == {"", *launches[2:]}


@pytest.mark.parametrize("tokens,hidden,experts,top_k,inter,kernels,gradients", [case for case in tiles.GROUPED + ragged.SHAPES])
def test_kernels_without_a_choice_of_tiles_name_themselves(tokens, hidden, experts, top_k, inter, kernels, gradients):
    names = product_tiles(tokens * top_k, hidden, inter, experts)
    for kernel, name in zip(kernels.split() + gradients.split(), names):
        assert (name == kernel) == (kernel.startswith(("stream", "rows64", "rows256_short")))


def test_sizes_out_of_range_have_no_tiles():
    assert product_tile(GATE_UP, 0, 64, 64) == product_tile(4, 1, 64, 64) == ""
    assert product_tile(GATE_UP, 1, 63, 64) == product_tile(DOWN, 1, 64, 12) == "general"
    assert joint_tiles(0, 2, 512, 512, 512, 8) == [""] * 4 and shared_beside(300, 9, 512, 512, 512, 8) == ["", ""]


@pytest.mark.parametrize("rows,hidden,inter,experts,names", [
    # what a taller tile spares against what it takes longer, by the measured sizes
    (64 * 512, 2048, 1408, 64, "plain tall tall tall"),
    (64 * 698, 2048, 1408, 64, "plain plain plain plain"),         # many rounds, hardly fewer tiles
    (64 * 1024, 2048, 1408, 64, "tall tall plain tall"),           # fewer tiles; seven rounds of dZ for six
    (128 * 688, 2048, 768, 128, "plain plain plain plain"),
    (24 * 698, 1000, 2664, 24, "plain_tail 128x256 plain_tail 128x128_pair"),
    (16 * 1375, 1024, 2816, 16, "tall plain plain plain"),         # five rounds for four of one data gradient
])
def test_taller_tiles_where_they_spare_more_than_they_cost(rows, hidden, inter, experts, names):
    assert product_tiles(rows, hidden, inter, experts) == names.split()


def test_taller_tiles_beside_dense_ones():
    assert joint_tiles(2621, 8, 2048, 1408, 2816, 64) == ["separate", "plain", "separate", "plain"]  # five rounds for four
    assert joint_tiles(2048, 8, 2048, 1408, 2816, 64)[0] == "tall"  # ... but with 3.4 rounds of tiles for 4.8
    assert joint_tiles(4096, 8, 2048, 1408, 2816, 64)[0] == joint_tiles(5588, 8, 2048, 1408, 2816, 64)[0] == "tall"


def with_tails(*names):
    return {name + tail for name in names for tail in ("", "_tail")}


LARGE = with_tails("tall", "plain")
GATE_UP_TILES = with_tails("64x64", "128x64", "128x128", "128x128_short") | LARGE
DOWN_TILES = {"64x64", "128x64", "128x128", "128x128_short", "128x128_pair", "256x128", "128x256"} | LARGE
GRADIENT_TILES = DOWN_TILES - {"128x128_short"}


def test_every_tile_is_held_to_the_bits_of_the_others():
    """... which the GPU test takes, by the rows of a dense call and by the tokens of a layer call."""
    alone, joint_ones = [set() for _ in range(4)], [set() for _ in range(4)]

    def add(sets, names):
        for seen, name in zip(sets, names):
            seen.add(name)

    for hidden, inter, rows in shapes.DENSE:
        for n in rows:
            add(alone, product_tiles(n, hidden, inter))
    for hidden, inter, shared, experts, top_k, tokens in shapes.LAYERS:
        for n in tokens:
            add(alone, product_tiles(n * top_k, hidden, inter, experts))
            if shared:
                add(alone, product_tiles(n, hidden, shared))
                add(joint_ones, joint_tiles(n, top_k, hidden, inter, shared, experts))
    for seen, names in zip(alone, (GATE_UP_TILES, DOWN_TILES, GRADIENT_TILES, GRADIENT_TILES)):
        assert seen >= names
    pair = {"128x128_pair"}
    for seen, names in zip(joint_ones, (GATE_UP_TILES, DOWN_TILES - pair, GRADIENT_TILES - pair, GRADIENT_TILES - pair)):
        assert seen == names | {"separate"}


@pytest.mark.parametrize("hidden,inter,tall_ones", tall.WIDTHS)
def test_rows_beyond_256_spare_a_round_of_the_products_named(hidden, inter, tall_ones):
    def mtiles(n, extra):  # as the kernels count them
        whole = max(1, n // 256)
        return whole + (n - whole * 256 > extra * whole) if n else 0

    names = product_tiles(sum(tall.SIZES), hidden, inter, len(tall.SIZES))
    columns = -(-inter // 128), -(-hidden // 256), -(-inter // 256), -(-hidden // 256)
    for product, (name, across) in enumerate(zip(names, columns)):
        plain, taller = (-(-across * sum(mtiles(n, extra) for n in tall.SIZES) // MI355X_CUS) for extra in (0, 64))
        assert (name.startswith("tall") and taller < plain) == (product in tall_ones)
