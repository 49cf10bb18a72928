"""What scans, packs, permutes and descriptor builds are given lies within the
scratch that their _scratch functions promise, on the CPU: every cleared
area, the tiles' aggregates, counts and sums, the partition's buffers and
counters, at the ends of each rule and over many lengths between them."""
import fake_hip

SCRIPT = r'''
import ctypes as C
SCRATCH = 1 << 46                       # never touched: nothing runs
end = SCRATCH
bad, seen = [], set()
case, width = None, 4

def area(what, p, nbytes):
    seen.add(what)
    if p and p >= SCRATCH and p + nbytes > end:
        bad.append((case, what, p + nbytes - end))

def on_launch(name, wgs, args):
    if "k_fill_u32" in name:
        area("fill", word(args, 0), 4 * word(args, 2))
    elif "k_tile_aggs" in name:
        area("aggregates", word(args, 3), width * wgs)
    elif "k_pack_count" in name:
        area("counts", word(args, 2), 4 * wgs)
    elif "k_part_hist" in name:
        area("histograms", word(args, 3), 1024 * wgs)
    elif "k_tile_scan" in name:
        area("status", word(args, 3), 8 * 256 * wgs)
    elif "k_partition" in name:
        n, clog = word(args, 4), word(args, 6, C.c_int)
        out = C.cast(args[3], C.POINTER(C.c_uint64))
        if "Local16" in name:
            area("blocks", out[0], 2 * n)
            area("blocks", out[1], width * n)
        elif width == 4:
            area("pairs", out[0], 8 * n)
        else:
            area("pairs", out[0], 4 * n)
            area("pairs", out[1], 8 * n)
        area("children", word(args, 9), 4 * (((n - 1) >> clog) * word(args, 11, C.c_int) + 1))
    elif "k_reduce" in name and "finish" not in name:
        area("partials", word(args, 2 if "strided" in name else 3), width * wgs)
        i = 6 if "strided" in name else 7
        Post.to(word(args, i), word(args, i + 1), 0)
    elif "k_segd_sums" in name:
        area("sums", word(args, 2), 8 * wgs)
    elif "k_segd_offsets" in name:
        area("count", word(args, 8), 4)

fake, lib = load(on_launch)
A, B, D = 1 << 43, 1 << 44, 1 << 45

def call(name, n, *args, size=None):
    global end, case
    end = SCRATCH + 8 * getattr(lib, name + "_scratch")(*(size or (n,)))
    case = (name, n)
    getattr(lib, name)(*args, SCRATCH)

lengths = list(range(1, 300)) + [k * 1021 for k in range(1, 200)]
for k in range(9, 29):
    lengths += [(1 << k) - 1, 1 << k, (1 << k) + 1, 3 << (k - 1), (3 << (k - 1)) + 1]
lengths += [20 << 20, (20 << 20) + 1, 49152, 49153]
for n in sorted(set(lengths)):
    for ty in "zd":
        width = 8 if ty == "d" else 4
        call(f"add_su{ty}", n, D, A, n)
        call(f"max_su{ty}", n, D, A, n)
        call(f"add_ru{ty}", n, A, n)
        call(f"pk2_lu{ty}", n, D, A, B, n, n // 2)
        call(f"smp_pu{ty}", n, D, A, B, n)
        call(f"dpe_pu{ty}", n, D, A, B, A, n // 3, n, size=(n // 3, n))
    for m in (1, 2, 4096, 4097, 100_000, 5_000_000):
        call("mke_fov", (n, m), D, A, n, m, size=(n, m))
assert seen == {"fill", "aggregates", "counts", "histograms", "status", "blocks", "pairs", "children", "partials", "sums",
                "count"}, seen
assert not bad, f"{len(bad)} areas past the scratch, bytes too many: {bad[:8]}"
print("ok")
'''


def test_areas_lie_within_the_promised_scratch(tmp_path):
    assert fake_hip.run(SCRIPT, tmp_path).startswith("ok")
