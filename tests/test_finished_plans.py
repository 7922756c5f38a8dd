"""What cuttPlan decides about a plan after the cost model has chosen it, without a GPU."""
import pytest

import fake_planner

TILED = 4


@pytest.fixture(scope="module")
def planner(tmp_path_factory):
    return fake_planner.build(tmp_path_factory.mktemp("planner"))


def test_pacing_is_part_of_the_plan(planner):
    # 8-byte batches off the line grid with output rows of 888 bytes: ordinary stores, below and above 0.75 cache sizes per buffer
    large, small = ((777, 111, 1000), (1, 0, 2), 8), ((777, 111, 200), (1, 0, 2), 8)
    assert [planner.plan(*large).tiledPaced, planner.plan(*small).tiledPaced] == [1, 0]
    assert planner.plan(*large).cachePolicy == 0
    # the option reaches plans of both sizes, also where the same tensor has been planned without it
    assert [planner.plan(*t, CUTT_TILED_PACED=0).tiledPaced for t in (large, small)] == [0, 0]
    assert [planner.plan(*t, CUTT_TILED_PACED=1).tiledPaced for t in (large, small)] == [1, 1]
    # past the caches, wide tiles, line-aligned stores: other kernels
    for dim, es in (((6000, 6080), 4), ((8192, 8192), 4), ((8200, 5003), 8)):
        assert planner.plan(dim, (1, 0), es).tiledPaced == 0
    assert planner.plan(*large, CUTT_CACHE_POLICY=3).tiledPaced == 0 and planner.plan(*large, CUTT_CACHE_POLICY=1).tiledPaced == 1


def test_blocks_are_those_of_the_launch(planner):
    # strips of tiles (8224 x 8192: 129 x 128 in strips of 8, the last one a tile wide): the kernels that decode a walk launch no padding
    # workgroups but the last XCD's, the general one all of the padded strips
    tiles = 129 * 128
    assert planner.plan((8224, 8192), (1, 0), 4, CUTT_XCD_GROUP=0).numBlocks == (tiles + 7) // 8 * 8
    assert planner.plan((8224, 8192), (1, 0), 4, CUTT_XCD_GROUP=5).numBlocks == (tiles + 127) // 128 * 128
    assert planner.plan((8224, 8192), (1, 0), 4, CUTT_XCD_GROUP=0, CUTT_TILED_PACED=1).numBlocks == 17 * 8 * 128
    # wide tiles: 65 x 64 in strips of 16
    assert planner.plan((8320, 8192), (1, 0), 4, CUTT_XCD_GROUP=0, CUTT_SUPER_M=16, CUTT_TILED_WIDE=1).numBlocks == (65 * 64 + 7) // 8 * 8


def test_groups_do_not_depend_on_who_chose_the_order(planner):
    # a pinned order is walked in the same groups as the planner's own
    for dim, perm, es in (((6000, 6080), (1, 0), 4), ((96, 75, 96, 75), (2, 1, 3, 0), 8), ((8200, 5003), (1, 0), 8)):
        own = planner.plan(dim, perm, es)
        assert own.xcdGroup == 5
        for env in (dict(CUTT_TILED_ORDER=own.tiledOrder), dict(CUTT_SUPER_M=8), dict(CUTT_SUPER_M=8, CUTT_SUPER_K=4096)):
            pinned = planner.plan(dim, perm, es, TILED, CUTT_TILED_ALIGNED=own.tiledAligned, **env)
            assert pinned.xcdGroup == 5, (dim, perm, es, env)


def test_whole_mm_axis_at_a_stretch_in_chunks_only(planner):
    # a fused Mm axis on the line grid: strips where the XCDs take groups
    dim, perm = (6, 320, 8, 4704), (3, 1, 2, 0)
    groups, chunks = planner.plan(dim, perm, 8), planner.plan(dim, perm, 8, CUTT_XCD_GROUP=0)
    assert (groups.xcdGroup, groups.tiledOrder, groups.superM) == (5, 3, 8)
    assert (chunks.xcdGroup, chunks.tiledOrder) == (0, 1)


def test_batches_with_few_rows_between_walk_strips_in_groups(planner):
    # (few rows between, many, no batch): patches 8 tiles along Mk everywhere but for the first in groups
    for dim, perm, strips in (((640, 11, 1344, 16), (2, 1, 0, 3), True), ((1088, 40, 1280, 3), (2, 1, 0, 3), False), ((1856, 67, 1280), (2, 1, 0), False)):
        tiles = (dim[2] + 63) // 64
        groups, chunks = planner.plan(dim, perm, 8), planner.plan(dim, perm, 8, CUTT_XCD_GROUP=0)
        assert (groups.xcdGroup, chunks.xcdGroup) == (5, 0)
        assert chunks.superK < tiles and (groups.superK == tiles) == strips, (dim, groups.superK, chunks.superK)


@pytest.mark.parametrize("dim,perm,es,group", [
    # output rows a multiple of 32 KB apart under 64x64 tiles; others; wide tiles
    ((8224, 8192), (1, 0), 4, 0), ((5040, 2, 8192), (2, 1, 0), 8, 0), ((8224, 8160), (1, 0), 4, 5), ((8192, 8192), (1, 0), 4, 5),
    # 8-byte rows of 64 KB beside 160 tiles along Mk and more, of 128 KB
    ((8192, 12352), (1, 0), 8, 0), ((16384, 10832), (1, 0), 8, 5), ((8192, 9200), (1, 0), 8, 5),
    # separate matrices off the line grid in strips, inside one cache size, in one strip, on the grid; without a batch
    ((2463, 128, 72), (1, 0, 2), 8, 5), ((1768, 64, 773), (1, 0, 2), 8, 0), ((979, 320, 558), (1, 0, 2), 4, 0), ((717, 448, 272), (1, 0, 2), 8, 5), ((512, 256, 667), (1, 0, 2), 8, 5),
    ((1768, 40976), (1, 0), 8, 5),
    # line-aligned stores: 4-byte strips, front to back; both axes over fused ranks without an Mbar rank, with one, one axis
    ((379, 131928), (1, 0), 4, 0), ((28309, 1348), (1, 0), 4, 5), ((60, 36, 2764, 3), (3, 2, 1, 0), 8, 0),
    ((14, 103, 1509, 9, 5), (3, 2, 1, 4, 0), 8, 5), ((62, 12, 42642), (2, 1, 0), 8, 5),
])
def test_plans_that_do_not_gain_in_groups(planner, dim, perm, es, group):
    info = planner.plan(dim, perm, es)
    assert info.method == TILED and info.xcdGroup == group


def test_matrices_in_strips_off_the_line_grid_are_paced(planner):
    # beyond one cache size per buffer, whatever their stores; not in one strip, not on the grid, not inside the cache
    for dim, es, paced in (((1822, 320, 150), 8, 1), ((981, 448, 398), 4, 1), ((717, 448, 272), 8, 0), ((512, 256, 667), 8, 0), ((2463, 128, 72), 8, 0)):
        info = planner.plan(dim, (1, 0, 2), es)
        assert (info.method, info.tiledPaced, info.cachePolicy & 2) == (TILED, paced, 2), dim
    assert planner.plan((1822, 320, 150), (1, 0, 2), 8, CUTT_TILED_PACED=0).tiledPaced == 0


CACHE = 256 << 20  # what the stand-in device reports


@pytest.mark.parametrize("dim,perm,es,policy", [
    # packed plans whose lines are written whole, on either side of a sixth of the cache per buffer
    ((16, 12, 32, 909), (2, 0, 1, 3), 8, 0), ((16, 12, 32, 912), (2, 0, 1, 3), 8, 2), ((16, 12, 32, 2600), (2, 0, 1, 3), 8, 2),
    # with 16 % and more of them covered partly: below a third of the cache, above
    ((26, 218, 12, 120), (1, 2, 0, 3), 8, 2), ((4, 6, 2071, 4, 10, 15), (4, 2, 0, 3, 1, 5), 4, 0),
    # Tiled plans that write whole lines, others
    ((512, 512, 21), (1, 0, 2), 8, 0), ((512, 512, 22), (1, 0, 2), 8, 2), ((2177, 2585), (1, 0), 8, 0), ((2177, 7177), (1, 0), 8, 0),
])
def test_cache_policy_of_tensors_up_to_half_a_cache_size(planner, dim, perm, es, policy):
    info = planner.plan(dim, perm, es)
    size = es
    for d in dim:
        size *= d
    assert 2 * size <= CACHE
    assert info.cachePolicy == policy, (info.method, info.wrPartialLines / (size / 128))


def test_a_pinned_cache_policy_is_the_one_plans_are_chosen_for(planner):
    # estimates of stores past the caches, and the preference for tiles in groups, only with such stores
    dim, perm = (129975, 177), (1, 0)
    assert [planner.plan(dim, perm, 4, **env).method for env in ({}, dict(CUTT_CACHE_POLICY=0), dict(CUTT_CACHE_POLICY=1))] == [3, TILED, TILED]
    dim, perm = (8, 4, 262144, 24), (2, 1, 3, 0)
    assert [planner.plan(dim, perm, 4, **env).method for env in ({}, dict(CUTT_CACHE_POLICY=3), dict(CUTT_CACHE_POLICY=0))] == [TILED, TILED, 3]


def test_packed_plans_give_way_to_tiles_that_write_whole_lines(planner):
    # beyond half a cache size, up to the margin; partly written lines, numberings by address bits, smaller tensors
    assert planner.plan((8, 4, 262144, 24), (2, 1, 3, 0), 4).method == TILED
    tiled, packed = (planner.plan((8, 4, 262144, 24), (2, 1, 3, 0), 4, m).usPredicted for m in (TILED, 3))
    assert packed < tiled < 1.18 * packed
    assert planner.plan((8, 4, 26214, 24), (2, 1, 3, 0), 4).method != TILED
    assert planner.plan((5, 7, 11, 13, 17, 1093), (4, 2, 0, 5, 1, 3), 4).method != TILED


@pytest.mark.parametrize("dim,perm,es,numbered", [
    # the digit at address bit 11 right below the three slowest binary ones, written and read side
    ((2, 4096, 512, 64), (0, 3, 1, 2), 4, True), ((16, 2, 1024, 8, 4, 128), (5, 4, 2, 1, 3, 0), 8, True), ((4, 1024, 512, 64), (3, 1, 0, 2), 8, True),
    # ... with sixteen elements per lane; further below
    ((16, 12288, 512), (0, 2, 1), 4, False), ((16, 8, 4, 128, 512, 8), (5, 1, 4, 0, 3, 2), 4, False), ((4, 4, 32768, 512), (0, 1, 3, 2), 4, False), ((4, 2, 4, 1024, 512, 8), (3, 1, 2, 5, 4, 0), 8, False),
])
def test_packed_plans_are_numbered_by_address_bit_11_or_take_groups(planner, dim, perm, es, numbered):
    info = planner.plan(dim, perm, es)
    assert info.method in (2, 3) and (bool(info.tileDigits), info.xcdGroup) == ((True, 0) if numbered else (False, 5))
    plain = planner.plan(dim, perm, es, CUTT_ADDRESS_BITS=0)
    assert not plain.tileDigits and plain.xcdGroup == 5


@pytest.mark.parametrize("dim,perm,es,waves,blocks", [
    # 8-byte blocks of 10 KB and more, up to 12000: twelve waves and fewer, more waves; more blocks; 4-byte elements
    ((2, 3, 6, 17, 5, 16, 3, 29, 15), (5, 4, 2, 7, 0, 6, 8, 1, 3), 8, 12, 1), ((122, 6, 25, 88, 11, 2), (2, 0, 3, 1, 4, 5), 8, 6, 1), ((28, 1019, 9, 273), (1, 2, 0, 3), 8, 14, 2),
    ((14, 36, 38, 3, 669), (2, 1, 3, 0, 4), 8, 7, 2), ((135, 3890, 2, 55, 2), (2, 4, 0, 3, 1), 8, 12, 2), ((32, 32, 7, 9, 12, 29, 3), (2, 6, 4, 0, 5, 1, 3), 4, 16, 4),
])
def test_8_byte_packed_plans_take_one_block_per_workgroup(planner, dim, perm, es, waves, blocks):
    info = planner.plan(dim, perm, es, CUTT_XCD_GROUP=0)
    assert info.method in (2, 3) and info.ldsBytes >= 10240
    assert (info.numThreads // 64, info.itemsPerBlock) == (waves, blocks)
    items = info.volMbar * info.numSplit * info.numSplit2
    assert info.numBlocks == ((items + blocks - 1) // blocks + 7) // 8 * 8
    # options that pin the number or the order
    more = blocks if blocks > 1 else 2
    assert planner.plan(dim, perm, es, CUTT_MAX_ITEMS=more).itemsPerBlock == more
    assert planner.plan(dim, perm, es, CUTT_ITEM_ORDER=0).itemsPerBlock == more


def test_a_numbering_by_address_bits_fits_the_blocks_per_workgroup(planner):
    for dim, perm, blocks in (((4, 8192, 1024), (0, 2, 1), 1), ((4, 1024, 512, 64), (3, 1, 0, 2), 2)):
        info, pinned = planner.plan(dim, perm, 8), planner.plan(dim, perm, 8, CUTT_MAX_ITEMS=blocks)
        assert info.itemsPerBlock == pinned.itemsPerBlock == blocks and info.tileDigits == pinned.tileDigits != b"" and info.numBlocks == pinned.numBlocks


def test_wide_tiles_are_estimated_as_the_small_ones_they_stand_for(planner):
    # (counted as tiles of 64 elements they seem to issue a quarter of the requests)
    for dim, perm in (((8192, 8192), (1, 0)), ((4096, 256, 64), (1, 0, 2)), ((256, 400, 512), (2, 1, 0))):
        wide = planner.plan(dim, perm, 4, TILED, CUTT_TILED_WIDE=1)
        small = planner.plan(dim, perm, 4, TILED, CUTT_TILED_WIDE=0)
        assert (wide.tiledWide, small.tiledWide, wide.volMm, wide.volMk) == (1, 0, small.volMm, small.volMk)
        assert abs(wide.usPredicted / small.usPredicted - 1) < 0.01, (dim, wide.usPredicted, small.usPredicted)
        assert (wide.rdLines, wide.wrLines, wide.rdInstr, wide.wrInstr) == (small.rdLines, small.wrLines, small.rdInstr, small.wrInstr)
