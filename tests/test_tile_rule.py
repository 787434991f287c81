"""The rules that pick a prefill GEMM's tiles (pick_gemm_tile, pick_gemm_mix), restated with the constants of the source, against measured
times: those the constants were fitted to, others, and the two ways in which the QKV projection writes the cache."""
import os
import re

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = open(os.path.join(ROOT, "seq2seqsharp_amd", "csrc", "tship_gpt.hip")).read()
TABLE = open(os.path.join(ROOT, "profiles", "prefill_gemm_tiles.txt")).read().split("\n")
UNITS = 256


def _numbers(pattern):
    m = re.search(pattern, SOURCE)
    assert m, pattern
    return [float(x) for x in m.groups()]


def _ceil(a, b):
    return -(-a // b)


def _rule():
    costs = [[float(x.rstrip("f")) for x in c.split(",")] for c in re.findall(r"\{([\d., f]+)\}", re.search(r"static const Cost costs\[\] = \{(\{11, 64.*?)\};", SOURCE, re.S).group(1))]
    mid_load, big_load = _numbers(r"\(c\.tile \? ([\d.]+)f : ([\d.]+)f\) \* tiles / \(rounds \* ncu\)")
    fixed, per_block, per_tile = _numbers(r"us \+= ([\d.]+)f \+ ([\d.]+)f \* \(float\)splits \+ ([\d.]+)f \* \(float\)\(c\.rows \* c\.cols\) / 64\.0f")

    def pick(K, N, rows):
        kt, nt, best = _ceil(K, 16), _ceil(N, 32), None
        for tile, tr, tc, a, b in costs:
            if tile == 0 and rows < 256:
                continue
            n = _ceil(rows, int(tr)) * _ceil(nt, int(tc))
            group = 4 if tile >= 20 else 8
            for splits in range(1, 5 if tile else 2):
                blocks = n * splits
                if splits > 1 and (blocks > UNITS or (splits - 1) * _ceil(kt, group * splits) * group >= kt):
                    continue
                rounds = _ceil(blocks, UNITS)
                us = rounds * (a + b * _ceil(kt, splits)) * (1 + (mid_load if tile else big_load) * blocks / (rounds * UNITS))
                if splits > 1:
                    us += fixed + per_block * splits + per_tile * tr * tc / 64
                if best is None or us < best[0]:
                    best = (us, int(tile) + (100 * splits if splits > 1 else 0))
        return best[1]
    return pick


def test_the_picked_tile_is_close_to_the_best_one():
    """Within 1 % on average, within 15 % but for one size in fifty."""
    pick, over = _rule(), []
    for line in TABLE:
        m = re.fullmatch(r"(\d+) x (\d+) (\d+): (.*)", line)
        if m:
            us = {int(t): float(v) for t, v in re.findall(r"(\d+):([\d.]+)", m.group(4))}
            over.append(us[pick(int(m.group(1)), int(m.group(2)), int(m.group(3)))] / min(us.values()) - 1)
    assert len(over) > 600 and np.mean(over) <= 0.01 and np.mean(np.array(over) > 0.15) <= 0.02, (np.mean(over), np.mean(np.array(over) > 0.15))


def _mix():
    """pick_gemm_mix: one launch of any tile, or two of different ones for the columns of whole rounds and the others."""
    table = lambda name, head: [[float(x.rstrip("f")) for x in c.split(",")] for c in re.findall(r"\{([\d., f]+)\}", re.search(r"static const Cost %s\[\] = \{(%s.*?)\};" % (name, head), SOURCE, re.S).group(1))]
    costs = [(int(t), int(r), int(c), a, b) for t, r, c, a, b in table("costs", r"\{11, 64") + table("wide", r"\{0, 256")]
    code = lambda c: c[0] or (0 if c[2] == 8 else 40 + c[2] // 2)
    mid_load, big_load = _numbers(r"\(c\.tile \? ([\d.]+)f : ([\d.]+)f\) \* tiles / \(rounds \* ncu\)")
    fixed, per_block, per_tile = _numbers(r"us \+= ([\d.]+)f \+ ([\d.]+)f \* \(float\)splits \+ ([\d.]+)f \* \(float\)\(c\.rows \* c\.cols\) / 64\.0f")
    second, gain = _numbers(r"rest\.us \+ ([\d.]+)f;\s+if \(us < mix\.us && us < ([\d.]+)f \* one\.us\)")
    (margin,) = _numbers(r"other\.cols && all\.us >= ([\d.]+)f \* other\.us")

    def us(c, kt, tiles, splits=1):
        blocks = tiles * splits
        rounds = _ceil(blocks, UNITS)
        t = rounds * (c[3] + c[4] * _ceil(kt, splits)) * (1 + (mid_load if c[0] else big_load) * blocks / (rounds * UNITS))
        return t + (fixed + per_block * splits + per_tile * c[1] * c[2] / 64 if splits > 1 else 0)

    def usable(kt, rows, widths):
        return [c for c in costs if c[0] or (rows >= 256 and (c[2] == 8 or (widths and kt % 2 == 0)))]

    def one(kt, nt, rows, widths=True, credit=0.0):
        best = (1e30, None)
        for c in usable(kt, rows, widths):
            tiles = _ceil(rows, c[1]) * _ceil(nt, c[2])
            for splits in range(1, 5 if c[0] else 2):
                group = 4 if c[0] >= 20 else 8
                if splits > 1 and (tiles * splits > UNITS or (splits - 1) * _ceil(kt, group * splits) * group >= kt):
                    continue
                t = us(c, kt, tiles, splits) - (credit if code(c) == 0 else 0)
                if t < best[0]:
                    best = (t, code(c) + (100 * splits if c[0] else 0))
        return best

    def mixed(kt, nt, rows, widths):
        single = one(kt, nt, rows, widths)
        best = (single[0], single[1], 0, 0)
        for c in usable(kt, rows, widths):
            rt, ct = _ceil(rows, c[1]), _ceil(nt, c[2])
            cols = rt * ct // UNITS * UNITS // rt
            if 1 <= cols < ct:
                rest = one(kt, nt - cols * c[2], rows, widths)
                t = us(c, kt, rt * cols) + rest[0] + second
                if t < best[0] and t < gain * single[0]:
                    best = (t, code(c) + (100 if c[0] else 0), cols * c[2], rest[1])
        return best

    def pick(K, N, rows):
        kt, nt = _ceil(K, 16), _ceil(N, 32)
        other, every = mixed(kt, nt, rows, False), mixed(kt, nt, rows, True)
        return other if other[2] and every[0] >= margin * other[0] else every
    return pick, one


def _lines(name, pattern):
    path = os.path.join(ROOT, "profiles", name)
    return [m.groups() for m in (re.fullmatch(pattern, line) for line in open(path).read().split("\n")) if m]


def test_the_projection_writes_whole_fragments_where_that_is_less():
    """The microseconds that the choice loses are a tenth of what always or never taking the 256 x 256 tile for them loses, at the sizes the
    line was drawn for and at others."""
    pick, one = _mix()
    slope, fixed = _numbers(r"whole_saves = can_fuse_kv \? std::max\(0\.0f, ([\d.e-]+)f \* \(float\)\(R \* 2 \* GD\) - ([\d.]+)f\)")
    lost = always = never = 0.0
    rows = _lines("prefill_qkv_cache_write.txt", r"(\d+) (\d+) (\d+), (\d+): ([+-][\d.]+), \((\d+), (\d+), (\d+)\) ([+-][\d.]+)")
    for K, N, columns, R, _, tile, cols, rest, other_us in rows:
        K, N, R, other_us = int(K), int(N), int(R), float(other_us)
        best = pick(K, N, R)
        assert best[1:] == (int(tile), int(cols), int(rest)), "measured with another choice"
        if best[1:] == (0, 0, 0):
            continue
        credit = max(0.0, slope * R * int(columns) - fixed)
        single = one(K // 16, N // 32, R, True, credit)
        whole = credit > 0 and single[1] == 0 and (not best[2] or best[0] >= single[0])
        lost += (0.0 if whole else other_us) - min(0.0, other_us)
        always -= min(0.0, other_us)
        never += max(0.0, other_us)
    assert len(rows) > 150 and 10 * lost <= min(always, never), (lost, always, never)


def test_the_pick_at_sizes_that_no_constant_was_fitted_to():
    """The up projection of models and prompts that are in none of the tables behind the constants: what pick_gemm_mix takes against every
    tile in one launch, microseconds of a layer.  Within 2.5 % of the launch's estimate on average."""
    pick, _ = _mix()
    over = []
    for K, N, R, times in _lines("prefill_gemm_other_sizes.txt", r"(\d+) x (\d+) (\d+): (.*)"):
        us = dict(re.findall(r"(\w+):([\d.]+)", times))
        over.append(float(us["pick"]) / pick(int(K), int(N), int(R))[0])
    assert len(over) > 60 and np.mean(over) <= 0.025, (len(over), np.mean(over), max(over))
