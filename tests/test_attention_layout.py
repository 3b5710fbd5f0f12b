"""A CPU model of how the attention (csrc/attention.hip) maps launches, workgroups and waves to query rows and K/V tile sets.

The automatic choice (launch_attn) gives one launch or two, each in one layout over some of the batch's heads: twelve-wave
workgroups of 384 consecutive rows of the (batch, head, row) range, each head's rows padded to Lq_pad (a multiple of 32; every head
of at least 384 rows); four-wave workgroups of 128 rows of one head; or split ones of 128, 64 or 32 rows of one head, whose
waves form three groups that share the keys out. The model restates the kernel's and the launcher's integer arithmetic
and checks, over many shapes, that every (batch, head, row) is stored by exactly one lane of one launch (and computed by all
three groups of a split workgroup), that a wave's 32 rows lie in one head, that a workgroup spans at most two heads with tile set
c holding the K/V head the waves of set c read, that the copying waves cover both sets, that the groups' tiles are the keys' tiles,
and that the XCD block remap is a permutation. Planted mistakes (the padding dropped, the head of the second set taken
from the first, a second launch that starts at the first head) fail it.
"""
import pytest

QB, FLAT_ROWS, KB, SPLIT, CUS = 128, 384, 32, 3, 256
FLAT, FOUR, SPLIT128, SPLIT64, SPLIT32 = 12, 4, -12, -6, -3  # rda_attn_waves' numbers
WAVES_OF_ROWS = {FLAT: 12, FOUR: 4, SPLIT128: 4, SPLIT64: 2, SPLIT32: 1}


def remap(blk, nblocks):
    xcd, run, rest = blk % 8, nblocks // 8, nblocks % 8
    return xcd * run + min(xcd, rest) + blk // 8


def choose(B, H, Lq, Lk, int8_qk=False, q_aligned=True):
    """launch_attn's automatic choice: [(layout, first head, heads)]."""
    heads, lq_pad = B * H, -(-Lq // 32) * 32
    split, long_keys = Lk > (SPLIT - 1) * KB and q_aligned, Lk > 23 * KB

    def layout(count, few):
        grid = lambda rows: count * -(-Lq // rows)  # noqa: E731
        if few and grid(32) <= CUS:
            return SPLIT32
        if few and grid(64) <= CUS:
            return SPLIT64
        if few and grid(QB) <= CUS and (not int8_qk or Lk > 27 * KB):
            return SPLIT128
        return FLAT if Lq >= FLAT_ROWS and 3 * -(-count * lq_pad // FLAT_ROWS) >= 2 * CUS else FOUR

    flat = -(-heads * lq_pad // FLAT_ROWS)
    if Lq >= FLAT_ROWS and flat > CUS and flat % CUS:
        whole = flat // CUS * CUS * FLAT_ROWS // lq_pad
        rest = layout(heads - whole, split and long_keys) if whole else FLAT if 3 * (flat % CUS) >= 2 * CUS else FOUR
        if Lk <= ((44 if int8_qk else 24) if rest == FLAT else (64 if int8_qk else 40)) * KB:
            return [(FOUR, 0, heads)]
        if rest != FLAT and whole:
            return [(FLAT, 0, whole), (rest, whole, heads - whole)]
        return [(rest, 0, heads)]
    return [(layout(heads, split and long_keys and 8 * heads * -(-Lq // QB) >= CUS), 0, heads)]


def waves(layout, H, Hkv, Lq, head0, heads, pad=True, second_from_first=False):
    """Yields (block, wave, group, b, h, q0, store, set, kv of set 0, kv of set 1, two) as the kernel computes them."""
    rep, nr = H // Hkv, WAVES_OF_ROWS[layout]
    if layout == FLAT:
        assert Lq >= FLAT_ROWS
        lq_pad = (Lq + 31) // 32 * 32 if pad else Lq
        rows = heads * lq_pad
        nblocks = (rows + FLAT_ROWS - 1) // FLAT_ROWS
        for block in range(nblocks):
            blk = remap(block, nblocks)
            g0 = blk * FLAT_ROWS
            bh0, bh1 = head0 + g0 // lq_pad, head0 + (min(g0 + FLAT_ROWS, rows) - 1) // lq_pad
            if second_from_first:
                bh1 = bh0
            kv = [(bh0 // H, (bh0 % H) // rep), (bh1 // H, (bh1 % H) // rep)]
            for wq in range(12):
                gw = g0 + 32 * wq
                store = gw < rows
                gc = gw if store else rows - 32
                bh = head0 + gc // lq_pad
                yield block, wq, 0, bh // H, bh % H, gc % lq_pad, store, bh - bh0, kv[0], kv[1], bh1 != bh0
    else:
        groups = SPLIT if layout < 0 else 1
        qblocks = -(-Lq // (32 * nr))
        nblocks = qblocks * heads
        for block in range(nblocks):
            bh, qblk = divmod(remap(block, nblocks), qblocks)
            bh += head0
            kv = (bh // H, (bh % H) // rep)
            for wave in range(nr * groups):
                grp, wq = divmod(wave, nr)
                # Every group reads a set of its own, of the workgroup's one head; the first one stores.
                yield block, wave, grp, bh // H, bh % H, (qblk * nr + wq) * 32, grp == 0, grp, kv, kv, False


def check(B, H, Hkv, Lq, launches, second_at_start=False, **mistake):
    rep = H // Hkv
    seen, computed = {}, {}
    for n, (layout, first, heads) in enumerate(launches):
        blocks = {}
        for block, wave, grp, b, h, q0, store, st, kv0, kv1, two in waves(layout, H, Hkv, Lq, 0 if second_at_start else first, heads, **mistake):
            assert 0 <= b < B and 0 <= h < H
            if layout >= 0:
                assert 0 <= st <= 1 and (st == 0 or two), "a wave reads the second set only where the workgroup has one"
                # The set this wave reads holds its own (batch, KV head).
                assert (kv0, kv1)[st] == (b, h // rep), "wave reads another head's K/V"
            else:
                assert st == grp and kv0 == (b, h // rep), "group reads another head's K/V"
                for row in range(q0, min(q0 + 32, Lq)):
                    computed.setdefault((n, b, h, row), set()).add(grp)
            blocks.setdefault(block, set()).add((b, h))
            if not store:
                continue
            for row in range(q0, min(q0 + 32, Lq)):  # the wave's rows q0 .. q0 + 31, each stored only below Lq
                assert (b, h, row) not in seen, f"row {(b, h, row)} computed twice"
                seen[b, h, row] = (n, block, wave)
        assert all(len(found) <= (2 if layout == FLAT else 1) for found in blocks.values()), "a workgroup spans more heads than it has sets"
    assert len(seen) == B * H * Lq, "some rows not computed"
    assert all(groups == {0, 1, 2} for groups in computed.values())


SHAPES = [(1, 24, 24, 4096), (1, 2, 2, 384), (2, 3, 1, 416), (1, 4, 2, 640), (1, 3, 3, 400), (2, 2, 1, 1000), (1, 1, 1, 513),
          (3, 5, 5, 777), (1, 2, 2, 300), (2, 4, 1, 77), (1, 8, 2, 4160), (4, 6, 3, 1536)]


@pytest.mark.parametrize("B,H,Hkv,Lq", SHAPES)
def test_every_row_once_and_sets_match_heads(B, H, Hkv, Lq):
    for layout in WAVES_OF_ROWS:
        if layout != FLAT or Lq >= FLAT_ROWS:
            check(B, H, Hkv, Lq, [(layout, 0, B * H)])


# Two launches: 24 heads x 9293 rows (21 in two whole rounds, 3 left), 53 + 7 heads, batch 2 with the second launch inside the second
# batch; one launch of each layout around them.
@pytest.mark.parametrize("B,H,Hkv,Lq,Lk,layouts", [(1, 24, 8, 9293, 9293, [FLAT, SPLIT128]), (1, 60, 60, 1800, 1500, [FLAT, SPLIT64]), (2, 48, 12, 1100, 2100, [FLAT, SPLIT64]),
                                                   (1, 24, 24, 4200, 4200, [FLAT, SPLIT32]), (1, 60, 60, 1800, 500, [FOUR]), (1, 24, 24, 4096, 4096, [FLAT]),
                                                   (1, 24, 24, 1101, 1101, [SPLIT128]), (4, 1, 1, 1000, 1152, [SPLIT32]), (1, 24, 24, 6500, 6500, [FLAT, FOUR])])
def test_automatic_choice_computes_every_row_once(B, H, Hkv, Lq, Lk, layouts):
    launches = choose(B, H, Lq, Lk)
    assert [layout for layout, _, _ in launches] == layouts
    check(B, H, Hkv, Lq, launches)


@pytest.mark.parametrize("int8_qk", [False, True])
def test_automatic_choice_limits(int8_qk):
    """Over a grid of shapes: the heads are covered in order, once; a split layout has more than 736 keys (int8-QK in 128-row workgroups:
    864), 16-byte aligned query rows and a grid of at most one workgroup per CU; in a call of one launch also 128-row workgroups for an
    eighth of the CUs; a second launch follows whole rounds of twelve-wave workgroups only."""
    seen = set()
    for B in (1, 2, 4):
        for H in (1, 2, 3, 8, 24, 31, 48, 60):
            for Lq in (1, 33, 100, 383, 384, 400, 1000, 1101, 2048, 3000, 4200, 9293, 99000):
                for Lk in (64, 65, 736, 737, 864, 865, 1300, 2049, 9293):
                    launches = choose(B, H, Lq, Lk, int8_qk)
                    assert [first for _, first, _ in launches] == [0, launches[0][2]][:len(launches)] and sum(n for *_, n in launches) == B * H
                    seen.add(tuple(layout for layout, *_ in launches))
                    for layout, _, heads in launches:
                        if layout < 0:
                            assert Lk > (864 if int8_qk and layout == SPLIT128 else 736)
                            assert heads * -(-Lq // (32 * WAVES_OF_ROWS[layout])) <= CUS
                            assert len(launches) == 2 or 8 * heads * -(-Lq // QB) >= CUS
                    if len(launches) == 2:
                        lq_pad = -(-Lq // 32) * 32
                        rounds = -(-B * H * lq_pad // FLAT_ROWS) // CUS * CUS * FLAT_ROWS
                        assert launches[0][0] == FLAT and launches[0][2] * lq_pad <= rounds < (launches[0][2] + 1) * lq_pad
                    assert all(layout > 0 for layout, *_ in choose(B, H, Lq, Lk, int8_qk, q_aligned=False))
    assert {(FOUR,), (FLAT,), (SPLIT128,), (SPLIT64,), (SPLIT32,), (FLAT, FOUR), (FLAT, SPLIT128)} <= seen


@pytest.mark.parametrize("Lk", [65, 96, 97, 128, 161, 737, 1101])
def test_key_groups_share_the_tiles_out(Lk):
    """Group j's i-th tile is tile 3 i + j: all tiles once, the partial one last in its group, the groups' counts at most one apart."""
    tiles = -(-Lk // KB)
    counts = [(tiles - j + SPLIT - 1) // SPLIT for j in range(SPLIT)]
    walked = [[SPLIT * i + j for i in range(counts[j])] for j in range(SPLIT)]
    assert sorted(sum(walked, [])) == list(range(tiles)) and min(counts) >= 1 and max(counts) - min(counts) <= 1
    assert walked[(tiles - 1) % SPLIT][-1] == tiles - 1


@pytest.mark.parametrize("nblocks", [256, 264, 8, 7, 1, 9, 216, 255, 1000, 1003])
def test_block_remap_is_a_permutation(nblocks):
    assert sorted(remap(b, nblocks) for b in range(nblocks)) == list(range(nblocks))
    for x in range(8):  # an XCD's blocks are consecutive
        run = [remap(b, nblocks) for b in range(x, nblocks, 8)]
        assert run == list(range(run[0], run[0] + len(run))) if run else nblocks <= x


def test_flat_configuration_is_one_round_of_whole_heads_per_xcd():
    """The attention configuration (24 heads x 4096 rows): 256 twelve-wave workgroups; XCD x (blocks x, x + 8, ...)
    covers 12288 consecutive rows, i.e. heads 3x .. 3x + 2."""
    heads_of_xcd = {}
    blocks = set()
    for block, wave, grp, b, h, q0, store, st, kv0, kv1, two in waves(FLAT, 24, 24, 4096, 0, 24):
        heads_of_xcd.setdefault(block % 8, set()).add(h)
        blocks.add(block)
    assert blocks == set(range(256))
    assert all(heads == {3 * x, 3 * x + 1, 3 * x + 2} for x, heads in heads_of_xcd.items())


@pytest.mark.parametrize("mistake,shape", [({"pad": False}, (1, 3, 3, 400)), ({"second_from_first": True}, (2, 3, 1, 416)),
                                           ({"second_from_first": True}, (1, 4, 2, 640)), ({"second_at_start": True}, (1, 60, 60, 1800))])
def test_model_catches_mistakes(mistake, shape):
    B, H, Hkv, Lq = shape
    launches = choose(B, H, Lq, 1500) if "second_at_start" in mistake else [(FLAT, 0, B * H)]
    with pytest.raises(AssertionError):
        check(*shape, launches, **mistake)
