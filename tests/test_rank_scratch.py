"""What a rank's kernels are given lies within the scratch that its _scratch
function promises, on the CPU: the counts of each tile (k_rank_hist writes a
row of 256 words and, on the first pass, two OR words per tile) and every
cleared area, over lengths up to 5000 and the ends of each rule above, plain
and segmented, with few segments and with enough for three and four digits
of segment numbers."""

import fake_hip

SCRIPT = r'''
import ctypes as C
SCRATCH = 1 << 46                       # never touched: nothing runs
bounds = [SCRATCH, SCRATCH]
bad, seen = [], set()
case = None

def area(what, p, nbytes):
    seen.add(what)
    if p and bounds[0] <= p and not p + nbytes <= bounds[1]:
        bad.append((case, what, p + nbytes - bounds[1]))

def on_launch(name, wgs, args):
    if "k_fill_u32" in name:
        area("fill", word(args, 0), 4 * word(args, 2))
    elif "k_rank_hist" in name:
        area("counts", word(args, 1), 1024 * wgs)
        area("children", word(args, 2), 1024 * wgs)
        area("or words", word(args, 3), 8 * wgs)
    elif "k_or_post" in name:
        Post.to(word(args, 5), word(args, 6), (1 << 12) - 1)
    elif "k_tile_scan" in name:
        area("scanned", word(args, 0), 1024 * word(args, 1))

fake, lib = load(on_launch)
lengths = list(range(1, 1100)) + list(range(1100, 5000, 37)) + [4096, 4097, 8192, 16384, 16385, 32768, 32769]
for edge in (1 << 19, 1 << 21, 1 << 22, 1 << 23, 1 << 24, 1 << 26):
    lengths += [edge - 1, edge, edge + 1]
for n in lengths:
    for ty in "zd":
        units = getattr(lib, f"rku_lu{ty}_scratch")(n)
        bounds[1] = SCRATCH + 8 * units
        case = (n, ty, "plain")
        getattr(lib, f"rku_lu{ty}")(1 << 44, 1 << 45, n, SCRATCH)
        for m in (2, 300, 70_000, 17_000_000):
            bounds[1] = SCRATCH + 8 * getattr(lib, f"rkd_le{ty}_scratch")(n, m)
            case = (n, ty, m)
            getattr(lib, f"rkd_le{ty}")(1 << 44, 1 << 45, 1 << 43, n, m, SCRATCH)
assert {"fill", "counts", "or words"} <= seen, seen
assert not bad, f"{len(bad)} areas past the scratch, bytes too many: {bad[:8]}"
print("ok", len(lengths))
'''


def test_rank_areas_lie_within_the_promised_scratch(tmp_path):
    assert fake_hip.run(SCRIPT, tmp_path).startswith("ok")
