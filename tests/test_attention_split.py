"""A CPU model of the split-key attention layouts (attn_kernel with three key groups, csrc/attention.hip): what each wave of a
workgroup reads and writes in LDS between which barriers.

A workgroup is three groups of NR waves; group j walks tiles j, j + 3, ... through three LDS stages of its own set of tiles.
Restated from the kernel: the copies of a group's first two tiles; Q's rows, copied by all groups into the stages that the groups'
third tiles will fill; a barrier, the Q reads, a barrier; the steps, of which all but the last two copy a tile and end with a barrier;
for a group with a tile fewer, a barrier more; a barrier, after which groups 1 and 2 leave their results in LDS; a barrier, after
which group 0 adds them up and turns its output rows around in LDS.

Checked, for every layout, fp16 and int8 tiles, and every number of tiles from 3 to 20: all waves meet the same number of barriers; two
accesses of different waves to overlapping bytes with no barrier between them are both reads; a read finds the data that it
expects (its tile, its rows of Q, its results), complete (copies are waited for ahead of a barrier); everything lies inside the
workgroup's LDS. Planted mistakes (no extra barrier, Q staged where the second tile goes, no barrier after the Q reads, none before
the results are left, a tile copied one stage early) each fail.
"""
import pytest

KB, NS, LAYOUTS = 32, 3, (4, 2, 1)
MERGE_BYTES = 64 * 64 * 4 + 64 * 8


class Wave:
    """One wave's accesses, each with the number of barriers met before it."""

    def __init__(self, name):
        self.name, self.phase, self.log, self.pending = name, 0, [], []

    def read(self, start, size, expect):
        self.log.append((self.phase, "r", start, size, expect, self.phase))

    def write(self, start, size, data):
        self.log.append((self.phase, "w", start, size, data, self.phase))

    def copy(self, start, size, data):  # in flight from here to the next wait
        self.pending.append((self.phase, start, size, data))

    def wait(self):
        self.log += [(phase, "w", start, size, data, self.phase) for phase, start, size, data in self.pending]
        self.pending = []

    def barrier(self):
        self.phase += 1


def run(NR, all_tiles, int8_qk, extra_barrier=True, q_stage=2, q_barrier=True, merge_barrier=True, copy_ahead=2):
    k_row = 128 if int8_qk else 256
    k_bytes, v_bytes = KB * k_row + (256 if int8_qk else 0), KB * 256
    ks, vs = NS * k_bytes, NS * v_bytes
    voff = 3 * ks
    lds = max(3 * NS * (k_bytes + v_bytes), (NS - 1) * NR * MERGE_BYTES)
    counts = [(all_tiles - j + NS - 1) // NS for j in range(NS)]
    first = [((1 - n) % 3 + 3) % 3 for n in counts]
    waves = [Wave((grp, wq)) for grp in range(NS) for wq in range(NR)]

    def q_rows(wq):  # where the rows of wave wq of every group are staged: two halves of 16 rows
        at = lambda j: (first[j] + q_stage) % 3  # noqa: E731
        start = voff + at(wq) * vs + wq * v_bytes if wq < NS else at(0) * ks
        return start, start + 4096 if wq < NS else at(1) * ks + k_bytes

    for w in waves:
        grp, wq = w.name
        n = counts[grp]
        tile = lambda i: (first[grp] + i) % 3  # noqa: B023, E731 -- the stage of the group's i-th tile

        def issue(i, stage):  # the wave's share of a tile: its DMAs of K rows, of scales and of V rows
            kst, vst = stage * ks + grp * k_bytes, voff + stage * vs + grp * v_bytes  # noqa: B023
            for d in range(4 if int8_qk else 8):
                if d % NR == wq:  # noqa: B023
                    w.copy(kst + d * 1024, 1024, ("K", grp, i))  # noqa: B023
            if int8_qk and wq == 0:  # noqa: B023
                w.copy(kst + KB * 128, 256, ("K", grp, i))  # noqa: B023
            for d in range(8):
                if d % NR == wq:  # noqa: B023
                    w.copy(vst + d * 1024, 1024, ("V", grp, i))  # noqa: B023

        def read_k(i):
            w.read(tile(i) * ks + grp * k_bytes, k_bytes, ("K", grp, i))  # noqa: B023

        def read_v(i):
            w.read(voff + tile(i) * vs + grp * v_bytes, v_bytes, ("V", grp, i))  # noqa: B023

        issue(0, tile(0))
        if n > 1:
            issue(1, tile(1))
        for d in range(grp, 8, NS):
            w.copy(q_rows(wq)[d // 4] + d % 4 * 1024, 1024, ("Q", wq))
        w.wait()
        w.barrier()
        for start in q_rows(wq):
            w.read(start, 4096, ("Q", wq))
        if q_barrier:
            w.barrier()
        read_k(0)
        for i in range(n):
            steady = i < n - 2
            if steady:
                issue(i + 2, tile(i + copy_ahead))
            if i < n - 1:
                read_k(i + 1)
            read_k(i)  # settle, where the maximum moves
            read_v(i)
            if steady:
                w.wait()
                w.barrier()
        assert tile(n - 1) == 0 and (n == 1 or tile(n - 2) == 2), "the last steps' stages are constants"
        if extra_barrier and max(n - 2, 0) < max(max(counts) - 2, 0):
            w.barrier()
        if merge_barrier:
            w.barrier()
        if grp > 0:
            w.write(((grp - 1) * NR + wq) * MERGE_BYTES, MERGE_BYTES, ("O", grp, wq))
        w.barrier()
        if grp == 0:
            for j in range(NS - 1):
                w.read((j * NR + wq) * MERGE_BYTES, MERGE_BYTES, ("O", j + 1, wq))
            w.write(wq * MERGE_BYTES, 32 * 256, ("turn", wq))
            w.read(wq * MERGE_BYTES, 32 * 256, ("turn", wq))
        assert not w.pending
    return waves, lds


def errors(waves, lds):
    found = []
    if len({w.phase for w in waves}) != 1:
        return ["waves meet different numbers of barriers"]
    log = [(w.name, n, *entry) for w in waves for n, entry in enumerate(w.log)]
    writes = [e for e in log if e[3] == "w"]
    overlap = lambda a, b: a[4] < b[4] + b[5] and b[4] < a[4] + a[5]  # noqa: E731
    for a in log:
        if a[4] < 0 or a[4] + a[5] > lds:
            found.append(f"{a} outside {lds} bytes")
        for b in writes:  # a is open from phase a[2] to a[7] (a copy: until its wait)
            if a[0] != b[0] and overlap(a, b) and a[2] <= b[7] and b[2] <= a[7]:
                found.append(f"{a} and {b} with no barrier between them")
    for r in log:
        if r[3] != "r":
            continue
        covered = {}
        for b in writes:
            before = b[7] < r[2] if b[0] != r[0] else (b[7], b[1]) < (r[2], r[1])
            if before and overlap(r, b):
                for byte in range(max(r[4], b[4]), min(r[4] + r[5], b[4] + b[5]), 256):
                    covered[byte] = max(covered.get(byte, (-1, -1, None)), (b[7], b[1], str(b[6])))
        if len(covered) < r[5] // 256 or any(data != str(r[6]) for _, _, data in covered.values()):
            found.append(f"{r} finds {sorted({d for _, _, d in covered.values()})} in {len(covered)} pieces")
    return found


@pytest.mark.parametrize("int8_qk", [False, True])
@pytest.mark.parametrize("NR", LAYOUTS)
def test_split_layout_is_race_free(NR, int8_qk):
    for all_tiles in range(3, 21):
        assert errors(*run(NR, all_tiles, int8_qk)) == [], all_tiles


@pytest.mark.parametrize("mistake", [dict(extra_barrier=False), dict(q_stage=1), dict(q_barrier=False), dict(merge_barrier=False), dict(copy_ahead=1)])
@pytest.mark.parametrize("NR", LAYOUTS)
def test_model_catches_mistakes(NR, mistake):
    assert any(errors(*run(NR, all_tiles, False, **mistake)) for all_tiles in (10, 11, 13))
