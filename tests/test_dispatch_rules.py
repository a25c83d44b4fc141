"""The rules that choose between kernels, asked on the host (no GPU call is made): the objects that the library was linked
from, linked once more with a program that calls the rules themselves."""
import glob
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PACKAGE = os.path.join(ROOT, "jax-gpt_amd")
GATEUP, DOWN = 0, 1


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    objects = sorted(glob.glob(os.path.join(PACKAGE, "build", "*.o")))
    if not os.path.exists(hipcc) or not objects:
        pytest.skip("needs hipcc and the library's objects")
    exe = str(tmp_path_factory.mktemp("rules") / "rules")
    flags = ["--offload-arch=gfx950", "-O1", "-std=c++17", "-w", "-I", os.path.join(ROOT, "include"), "-I", os.path.join(PACKAGE, "csrc")]
    subprocess.run([hipcc, *flags, "-c", os.path.join(ROOT, "tests", "dispatch_rules.hip"), "-o", exe + ".o"], check=True)
    subprocess.run([hipcc, "--offload-arch=gfx950", exe + ".o", *objects, "-o", exe], check=True)

    def run(*commands):
        text = "\n".join(" ".join(str(int(v) if isinstance(v, bool) else v) for v in c) for c in commands)
        return subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.splitlines()
    return run


def test_ring_depth_follows_the_items_that_there_are(ask):
    """Short row tiles: one weight stage where all items run at once and some CUs have two, two stages otherwise -- by the
    list's items, not by what they could be at most (12 of 32 experts with rows: 192 items of at most 512)."""
    items = [192, 256, 257, 512, 513, 2048]
    assert ask(*[("depth", GATEUP, True, n // 16, n, n // 8) for n in items]) == ["2", "2", "1", "1", "2", "2"]
    # down, lists with taller tiles: by the rows of a tile
    assert ask(*[("depth", DOWN, False, 24, 672, r) for r in (24, 240, 241, 700)]) == ["2", "2", "1", "1"]
    assert ask(("depth", DOWN, True, 24, 672, 700)) == ["2"]


def test_lists_are_cut_for_the_kernels_that_read_them(ask):
    """128-row tiles are for the down GEMM's short-tile kernel: a list that a gate/up launch alone reads has none."""
    def rows(R, ncb, kb, E=32, most=None, dense=(0, 0, 0)):
        return ("tile_rows", R, E, R if most is None else most, *ncb, *kb, *dense)
    gateup, down, both = ((16, 0), (56, 0)), ((0, 28), (0, 16)), ((16, 28), (56, 16))
    for R, want in ((64, ("32", "32", "32")), (128, ("32", "32", "32")), (129, ("288", "128", "128")), (512, ("288", "128", "128")),
                    (513, ("288", "288", "288")), (16384, ("288", "288", "288"))):
        assert tuple(ask(rows(R, *gateup), rows(R, *down), rows(R, *both))) == want, R
    # too few items of the down GEMM for that kernel, whatever the gate/up GEMM has
    assert ask(rows(512, (16, 2), (4, 16), E=64)) != ["128"]
    # most rows of a group, and a shared expert beside
    assert ask(rows(256, (6, 8), (16, 6), E=128, most=32), rows(1024, (6, 8), (16, 6), E=128, most=128),
               rows(672, *both, E=256, most=84, dense=(84, 16, 28))) == ["32", "128", "32"]


def test_tall_tiles_are_for_even_groups_of_short_k_in_few_rounds(ask):
    """320 rows where the largest of even groups have more rows than whole full tiles and no more than whole tall ones."""
    from tests.test_gpu_variants import TALL, test_tall_tiles_give_the_bits_of_full_ones as tall

    def rows(R, E, D, I, dense=(0, 0, 0)):
        return ("tile_rows", R, E, R, I // 128, -(-D // 256), D // 128, I // 128, *dense)
    cases, = [m.args[1] for m in tall.pytestmark if m.name == "parametrize"]
    E, D, I = TALL.values()
    assert ask(*[rows(sum(c[i % len(c)] for i in range(E)), E, D, I) for c in cases]) == ["320"] * len(cases)
    assert ask(*[("voted", E, *(c[i % len(c)] for i in range(E))) for c in cases]) == ["320", "320", "320", "288", "288", "320"]
    even = {3500: "288", 3840: "288", 3860: "320", 4096: "320", 4400: "320", 4600: "288", 8000: "288", 8192: "320", 20000: "288"}
    assert ask(*[rows(8 * M, 128, 2048, 768) for M in even]) == list(even.values())
    # long K (twice), a dense group beside, more rounds
    assert ask(rows(65536, 256, 7168, 2048), rows(32768, 128, 2176, 768), rows(32768, 128, 2048, 768, (4096, 6, 8)),
               rows(131072, 512, 2048, 1024)) == ["288"] * 4
    # a list of one GEMM has none
    assert ask(("tile_rows", 32768, 128, 32768, 6, 0, 16, 0, 0, 0, 0), ("tile_rows", 32768, 128, 32768, 0, 8, 0, 6, 0, 0, 0)) == ["288", "288"]


def test_few_tokens_go_straight_to_their_experts_where_that_is_cheaper(ask):
    """By the weights read, those read again, and the second launch's chain: not a wide shared expert beside small routed
    ones, nor sixteen tokens that all read the same few experts."""
    taken = [(1, 7168, 256, 8, 2048, 2048), (8, 2048, 128, 8, 768, 0), (2, 4096, 512, 10, 1024, 1024), (16, 1024, 32, 2, 512, 512), (16, 512, 8, 2, 1024, 0),
             (4, 1024, 32, 2, 512, 4096), (4, 4096, 4, 2, 1024, 0), (8, 2048, 32, 8, 768, 0), (8, 1024, 8, 8, 1024, 0), (16, 512, 16, 16, 512, 0)]
    left = [(2, 7168, 256, 8, 2048, 2048), (9, 2048, 128, 8, 768, 0), (3, 4096, 512, 10, 1024, 1024), (17, 1024, 32, 2, 512, 512),
            (12, 1024, 32, 2, 512, 4096), (16, 1024, 32, 2, 256, 4096), (8, 4096, 4, 2, 1024, 0), (8, 4096, 2, 2, 1024, 1024), (12, 1024, 8, 8, 1024, 0), (12, 768, 8, 8, 1536, 0)]
    assert ask(*[("token", *c) for c in taken]) == ["1"] * len(taken)
    assert ask(*[("token", *c) for c in left]) == ["0"] * len(left)


def test_two_k_steps_a_stage_are_for_workgroups_that_run_at_once(ask):
    """From the caches as many as the CUs' LDS holds, from memory and of short rows four a CU; whole pairs of K steps only.  The
    batches that test_gpu_variants.py compares are on both sides of each."""
    from tests.test_gpu_variants import test_single_tokens_in_stages_of_one_and_two_k_steps as compared
    batches, = [m.args[1] for m in compared.pytestmark if m.name == "parametrize"]
    assert ask(*[("token", *c) for c in batches]) == ["1"] * len(batches)
    assert ask(*[("stages", *c) for c in batches]) == ["2 1", "1 1", "2 2", "1 2", "1 1", "1 2", "1 2"]
    limits = {(4, 2048, 32, 8, 768, 0): "2", (6, 2048, 32, 8, 768, 0): "1", (4, 1024, 8, 8, 1024, 0): "2", (8, 1024, 8, 8, 1024, 0): "1",   # 1536, 2304, 2048, 4096 workgroups
              (8, 512, 8, 2, 1024, 0): "2", (9, 512, 8, 2, 1024, 0): "1",                        # of short rows 1024, 1152
              (2, 2048, 128, 8, 768, 0): "2", (3, 2048, 128, 8, 768, 0): "1"}                    # from memory 768, 1152
    assert [a[0] for a in ask(*[("stages", *c) for c in limits])] == list(limits.values())


def test_single_tokens_are_routed_by_workgroups_that_run_at_once(ask):
    """Up to 256 experts and as many workgroups as the CUs' LDS holds; behind a small router about one a CU, two without a norm.  The
    batches that test_gpu_variants.py compares are on both sides."""
    from tests.test_gpu_variants import FRONTED_TOKENS, ROUTED_TOKENS
    assert ask(*[("token", *c) for c in ROUTED_TOKENS]) == ["1"] * len(ROUTED_TOKENS)
    assert ask(*[("token_routes", *c) for c in ROUTED_TOKENS]) == ["1"] * 5 + ["0", "1", "1", "1"]
    assert ask(*[("token", *c[:6]) for c in FRONTED_TOKENS]) == ["1"] * len(FRONTED_TOKENS)
    assert ask(*[("front", c[0], c[1], c[2], c[2] + (c[5] > 0), int(c[6]), 0, 1) for c in FRONTED_TOKENS]) == ["1"] * len(FRONTED_TOKENS)
    assert ask(*[("token_fronts", *map(int, c)) for c in FRONTED_TOKENS]) == ["1", "1", "1", "0", "1", "1", "1", "1", "1"]
    limits = {(1, 7168, 256, 8, 2048, 2048): "1", (8, 2048, 128, 8, 768, 0): "1", (1, 4096, 512, 10, 1024, 0): "0"}
    assert ask(*[("token_routes", *c) for c in limits]) == list(limits.values())
    assert ask(*[("token_selected", *c) for c in limits]) == ["1", "1", "1"]   # (whatever the experts' number)
    assert ask(("token_fronts", 6, 1024, 32, 2, 512, 512, 0), ("token_fronts", 1, 1024, 64, 2, 1152, 0, 1)) == ["0", "0"]   # 576 workgroups; from memory


def test_long_selections_are_not_repeated_by_many_workgroups(ask):
    """Ready logits: as many workgroups as 48 K steps of selection (64 or 128 K from D 1024 on), a step more for each group that lies across
    lanes, and one and a half for each of the grouped routing."""
    softmax, grouped = 0, 1
    want = {(16, 512, 256, 8, 512, 0, softmax, 1, 1): "1",      # 4096 workgroups, 32 K steps
            (6, 512, 64, 32, 128, 0, softmax, 1, 1): "1",       # 1536, 48 K
            (7, 512, 64, 32, 128, 0, softmax, 1, 1): "0",
            (16, 512, 64, 32, 128, 0, softmax, 1, 1): "0",
            (16, 512, 256, 8, 512, 0, grouped, 8, 4): "1",      # 48 K
            (4, 512, 64, 32, 128, 0, grouped, 8, 4): "1",       # 1024, 48 K
            (5, 512, 64, 32, 128, 0, grouped, 8, 4): "0",
            (2, 512, 240, 8, 512, 0, grouped, 48, 24): "1",     # groups of five: 512 workgroups, 42 K
            (3, 512, 240, 8, 512, 0, grouped, 48, 24): "0",
            (16, 512, 240, 8, 512, 0, grouped, 48, 24): "0",
            (16, 512, 240, 8, 512, 0, grouped, 48, 48): "1",    # (all groups are kept: nobody looks at them)
            (2, 512, 192, 8, 512, 0, grouped, 0, 0): "1",       # (refused later)
            (16, 1024, 256, 32, 128, 0, softmax, 1, 1): "1", (8, 1024, 64, 32, 128, 0, softmax, 1, 1): "1", (9, 1024, 64, 32, 128, 0, softmax, 1, 1): "0",
            (10, 1024, 256, 32, 128, 0, grouped, 8, 4): "1", (11, 1024, 256, 32, 128, 0, grouped, 8, 4): "0",   # longer rows stream meanwhile
            (1, 7168, 256, 8, 2048, 2048, grouped, 8, 4): "1", (8, 2048, 128, 8, 768, 0, softmax, 1, 1): "1"}
    assert ask(*[("token_chain", *c) for c in want]) == list(want.values())


def test_wider_routers_are_repeated_by_one_workgroup_a_cu(ask):
    """Behind a router the limit of workgroups is 256 where its weights are many; the batches that test_gpu_variants.py compares and
    the mini layer's 3 (behind its norm) and 5 tokens are on the same sides as without that line."""
    from tests.test_gpu_variants import FRONTED_TOKENS
    assert ask(*[("token_router", *map(int, c)) for c in FRONTED_TOKENS]) == ask(*[("token_fronts", *map(int, c)) for c in FRONTED_TOKENS])
    want = {(3, 1024, 64, 4, 256, 256, 0): "1", (3, 1024, 64, 4, 256, 256, 1): "1",      # 240 workgroups
            (4, 1024, 64, 4, 256, 256, 0): "0", (4, 1024, 64, 4, 256, 256, 1): "0",      # 320, 65 K weights
            (6, 768, 55, 4, 256, 256, 0): "1", (6, 768, 56, 4, 256, 256, 0): "0",        # 42 K and more
            (4, 512, 67, 4, 256, 256, 1): "1", (4, 512, 68, 4, 256, 256, 1): "0",        # 34 K
            (3, 1024, 32, 2, 512, 512, 1): "1", (5, 1024, 32, 2, 512, 512, 0): "1"}
    assert ask(*[("token_router", *c) for c in want]) == list(want.values())


def test_the_down_gemm_of_short_k_has_a_list_of_its_own(ask):
    """Tiles of 128 rows beside gate/up's full ones: more rows than one workgroup sorts, few K steps, enough items and not too many rows."""
    from tests.test_gpu_variants import TWO_LISTS
    want = {(256, 2048, 128, 8, 768, 0): "128 0", (257, 2048, 128, 8, 768, 0): "288 128", (3200, 2048, 128, 8, 768, 0): "288 128", (3201, 2048, 128, 8, 768, 0): "288 0",
            (4096, 2048, 128, 8, 768, 0): "320 0", (819, 4096, 512, 10, 1024, 1024): "128 0", (820, 4096, 512, 10, 1024, 1024): "288 128",
            (3276, 4096, 512, 10, 1024, 1024): "288 128", (3277, 4096, 512, 10, 1024, 1024): "288 0", (777, 7168, 256, 8, 2048, 2048): "288 0",
            (2000, 2048, 128, 8, 1152, 0): "288 0"}
    assert ask(*[("down_list", *c) for c in want]) == list(want.values())
    assert ask(*[("down_list", *c[:6]) for c in TWO_LISTS]) == ["288 128"] * len(TWO_LISTS)


def test_scales_are_placed_with_their_rows_where_they_are_few(ask):
    """The batches that test_gpu_variants.py compares: placed, or by a launch of their own; beside two work lists one of each kind, and their
    parts, which one workgroup sorts, read them in place."""
    from tests.test_gpu_variants import PLACED, TWO_LISTS
    assert ask(*[("scales", M, D, 12, 2, 128, 0) for M, D in PLACED]) == ["1 1"] * 4 + ["1 0"] * 2
    assert ask(*[("scales", 500, D, 12, 2, 128, 0) for M, D in PLACED]) == ["0 0"] * 6
    assert ask(*[("scales", M, D, E, k, I, 0) for M, D, E, k, I, SI, offset in TWO_LISTS]) == ["0 0", "1 0", "1 1", "0 0", "0 0"]
    assert ask(("scales", 8192, 2048, 12, 2, 128, 1), ("scales", 4096, 2048, 128, 8, 768, 0), ("scales", 2000, 2048, 128, 8, 768, 0),
               ("scales", 777, 7168, 256, 8, 2048, 0), ("scales", 1024, 2048, 128, 8, 768, 0)) == ["1 0", "1 0", "1 1", "1 0", "0 0"]


def test_selections_that_a_quantiser_goes_in_front_of(ask):
    """The dropped entries that test_gpu_variants.py compares: read by the launch that quantises too, and by the one that does not."""
    from tests.test_gpu_variants import DROPPED
    inside = [(M, 512, 10, k, 256, 0) for M, k in ((1, 2), (5, 3), (16, 8))]
    assert ask(*[("token", *c) for c in inside + [DROPPED]]) == ["1"] * 4
    assert ask(*[("token_selected", *c) for c in inside + [DROPPED]]) == ["1", "1", "1", "0"]


def test_a_shared_expert_of_long_k_keeps_the_list_of_tall_tiles(ask):
    """Where one item of its short tiles would outlast the launch; not where it is one tall tile, or most of the work, or where the
    routed experts' items take as long."""
    want = {(384, 2048, 128, 8, 768, 2048): True, (384, 2048, 128, 8, 768, 3072): False, (640, 2048, 128, 8, 768, 3072): True,
            (384, 2048, 128, 8, 768, 6144): False, (1200, 2048, 128, 8, 768, 6144): False, (1440, 2048, 128, 8, 768, 6144): True,
            (272, 2048, 128, 8, 768, 6144): True, (544, 4096, 256, 8, 512, 4096): True,
            (640, 1024, 256, 8, 512, 4096): False, (384, 2048, 128, 8, 768, 0): True, (2047, 4096, 512, 10, 1024, 1024): True}
    assert [int(a.split()[1]) > 0 for a in ask(*[("down_list", *c) for c in want])] == list(want.values())


def test_small_layers_read_the_selection_themselves(ask):
    """Few rows of few experts from the caches, in tiles of up to 128 rows; not where a list's tiles are taller for a reason, nor
    where the short-tile kernel takes the launch."""
    from tests.test_gpu_variants import SCANNED
    assert all(32 <= int(r) <= 128 for r in ask(*[("scan", *c[:6]) for c in SCANNED]))
    assert ask(*[("token", *c[:6]) for c in SCANNED]) == ["0"] * len(SCANNED)
    left = [(1025, 512, 8, 2, 1024, 0), (100, 512, 65, 2, 256, 0), (100, 4096, 32, 2, 2048, 0),   # rows, experts, weights from memory
            (512, 4096, 2, 2, 4096, 0), (128, 1536, 64, 8, 256, 0)]                              # 512 rows an expert in tall tiles; 384 items of short ones
    assert ask(*[("scan", *c) for c in left]) == ["0"] * len(left)


def test_small_layers_down_launch_is_for_one_workgroup_a_cu(ask):
    """64 selections a workgroup where that is no more than 256, else 128, while a workgroup's rows are few; the batches that
    test_gpu_variants.py compares are of both kinds."""
    from tests.test_gpu_variants import SMALL_DOWN
    assert ask(*[("small", *c[:6]) for c in SMALL_DOWN]) == [str(c[6]) for c in SMALL_DOWN]
    assert all(int(r) for r in ask(*[("scan", *c[:6]) for c in SMALL_DOWN]))
    assert ask(*[("token", *c[:6]) for c in SMALL_DOWN]) == ["0"] * len(SMALL_DOWN)
    limits = {(256, 512, 8, 2, 1024, 0): "1", (257, 512, 8, 2, 1024, 0): "2", (512, 512, 8, 2, 1024, 0): "2", (513, 512, 8, 2, 1024, 0): "0",
              (128, 1024, 32, 2, 512, 512): "1", (256, 1024, 32, 2, 512, 512): "2", (257, 1024, 32, 2, 512, 512): "0",
              (96, 1024, 32, 2, 2048, 0): "0", (128, 1024, 32, 4, 1024, 0): "0",          # too much for one workgroup
              (33, 128, 4, 33, 128, 0): "0", (20, 128, 4, 2, 8320, 0): "0", (20, 128, 4, 2, 128, 8320): "0", (20, 128, 65, 2, 128, 0): "0"}
    assert ask(*[("small", *c) for c in limits]) == list(limits.values())


def test_small_layers_down_launch_is_for_few_units(ask):
    """By what a workgroup copies, 16 weight rows for every unit, which is more where many experts have a row or two each."""
    want = {(64, 256, 64, 2, 512, 1024): "0", (128, 256, 64, 2, 512, 512): "0", (128, 512, 64, 4, 640, 512): "0", (17, 512, 64, 2, 1024, 0): "0",
            (32, 512, 32, 4, 1024, 0): "0", (32, 256, 64, 8, 512, 0): "0", (32, 256, 64, 8, 256, 0): "1", (128, 1024, 32, 2, 512, 512): "1", (256, 1024, 32, 2, 512, 512): "2"}
    assert ask(*[("small", *c) for c in want]) == list(want.values())
    from tests.test_gpu_variants import UNITS
    assert ask(*[("small", sum(c) // k, D, E, k, I, SI) for c, D, E, k, I, SI in UNITS]) == ["1", "1", "2"]
    assert all(int(r) for r in ask(*[("scan", sum(c) // k, D, E, k, I, SI) for c, D, E, k, I, SI in UNITS]))


def test_the_compared_batches_of_single_tokens_reach_what_they_are_for(ask):
    """The batches that test_gpu_variants.py compares with the grouped route take the other one, and among them are: a last
    workgroup of fewer tiles, one over two scale blocks, more slots than waves, waves that LDS limits, weights from memory."""
    from tests.test_gpu_variants import test_experts_of_single_tokens_give_the_grouped_bits as single
    cases, = [m.args[1] for m in single.pytestmark if m.name == "parametrize" and "M,D" in m.args[0]]
    assert ask(*[("token", *c) for c in cases]) == ["1"] * len(cases)
    memory = [v == "1" for v in ask(*[("memory", E, D, I, SI) for M, D, E, k, I, SI in cases])]
    plans = [tuple(map(int, v.split())) for v in ask(*[("down", M, D, k, I, SI) for M, D, E, k, I, SI in cases])]
    reached = {"from memory": memory}
    reached["last workgroup"] = [D // 16 % t > 0 for (M, D, *_), (t, _, _) in zip(cases, plans)]
    reached["two scale blocks"] = [any(b * t % 8 + min(t, D // 16 - b * t) > 8 for b in range(-(-D // 16 // t))) for (M, D, *_), (t, _, _) in zip(cases, plans)]
    reached["sixteen waves"] = [w == 16 < k + (SI > 0) for (*_, k, I, SI), (_, w, _) in zip(cases, plans)]
    reached["lds"] = [bool(limited) for _, _, limited in plans]
    reached["several tokens from memory"] = [m and c[0] > 1 for m, c in zip(memory, cases)]
    assert all(map(any, reached.values())), reached
    assert {t for t, _, _ in plans} >= {1, 2, 3, 16}


def test_a_dense_group_beside_routed_rows_needs_their_list(ask):
    """Cut on its own it could have taller tiles than the kernel that the routed list's height chooses."""
    assert ask(("both",))[0].startswith("-1 -1 gemm_down: a dense group")


def test_small_routers_of_many_tokens_go_launch_by_launch(ask):
    """One workgroup a CU has 4096 tokens; more of them only where that is faster."""
    from tests.test_gpu_variants import test_small_routers_in_one_launch_give_the_bits_of_the_stages as small

    def takes(*calls):
        return ask(*[("front", M, D, E, E, *flags) for M, D, E, *flags in calls])
    norm, bare, f32, alone = (True, False, True), (False, False, True), (False, True, True), (False, False, False)
    # what test_gpu_variants.py compares: all of it in one launch, but for the norm of the largest batch
    compared, = [m.args[1] for m in small.pytestmark if m.name == "parametrize"]
    for M, D, E, SI, dtype, _ in compared:
        flags = [(has_norm, dtype == "f32", True) for has_norm in (True, False)] + [alone]
        assert ask(*[("front", M, D, E, E + (SI > 0), *f) for f in flags]) == ["0" if M > 4096 else "1", "1", "1"], (M, D, E)
    # too many experts, too long rows, rows of no whole blocks, K slices of more than one block
    assert takes((100, 512, 65, *norm), (100, 1152, 8, *norm), (100, 192, 8, *norm), (12000, 1024, 64, *alone)) == ["0"] * 4
    taken = [(4096, 1024, 64, *norm), (4096, 128, 8, *norm), (4097, 512, 64, *bare), (32768, 256, 64, *bare), (4600, 1024, 64, *f32), (4600, 1024, 64, *alone),
             (32768, 128, 64, *alone)]
    left = [(4097, 1024, 64, *norm), (4097, 128, 8, *norm), (65536, 128, 64, *norm), (4097, 640, 64, *bare), (32769, 128, 64, *bare), (32769, 128, 64, *alone),
            (262144, 128, 8, *alone)]
    assert takes(*taken) == ["1"] * len(taken)
    assert takes(*left) == ["0"] * len(left)


def test_routers_refuse_activations_beyond_4_gb_whatever_the_launch(ask):
    """128 columns and 64 experts go to the launch that has everything in one, 65 experts to the matmul's own."""
    for E in (64, 65):
        assert ask(("routing", 1 << 24, 128, E))[0].startswith("-1 router: the activations must stay within 4 GB"), E
