"""The tuner's longest pack tiles, on the CPU: the library builds with them,
and the counts of the shorter tiles that mid-size vectors are packed in lie
within the scratch, which the long tiles' status words alone would not fill."""
import fake_hip

SCRIPT = r'''
SCRATCH = 1 << 46
bad, seen = [], 0

def on_launch(name, wgs, args):
    global seen
    at, size = (word(args, 2), 4 * wgs) if "k_pack_count" in name else (
        (word(args, 0), 4 * word(args, 2)) if "k_fill_u32" in name else (0, 0))
    seen += "k_pack_count" in name
    if at + size > end:
        bad.append((n, name, at + size - end))

fake, lib = load(on_launch)
for n in [k * 997 for k in range(1, 400)] + [(1 << 22) + 1, (1 << 24) - 1, 1 << 24, (1 << 24) + 1, 1 << 26]:
    for ty in "zd":
        end = SCRATCH + 8 * getattr(lib, f"pk2_lu{ty}_scratch")(n)
        getattr(lib, f"pk2_lu{ty}")(1 << 43, 1 << 44, 1 << 45, n, n, SCRATCH)
assert seen and not bad, (seen, bad[:5])
print("ok")
'''


def test_long_pack_tiles(tmp_path):
    assert fake_hip.run(SCRIPT, tmp_path, lib=fake_hip.variant(tmp_path, "pack.hip", "CVLHIP_PACK_ROWS", 10)).startswith("ok")
