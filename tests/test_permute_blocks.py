"""The tuner's sizes of the partition's final blocks, on the CPU: with each
of them every length about the limit of the direct permute has a path (one
that leaves pairs for a second partition pass, or none)."""
import pytest

import fake_hip

SCRIPT = r'''
launched = []
fake, lib = load(lambda name, wgs, args: launched.append(name))
for log in (13, 14, 18, 20, 21, 22, 23, 24, 25, 26):
    for n in ((1 << log) - 1, 1 << log, (1 << log) + 1):
        for ty in "zd":
            launched.clear()
            getattr(lib, f"smp_pu{ty}")(1 << 44, 1 << 45, 1 << 46, n, 1 << 47)
            passes = sum("k_partition" in x for x in launched)
            assert passes != 1, (n, ty, launched)
            placed = [x for x in launched if "k_permute_direct" in x or "k_block_scatter" in x]
            assert len(placed) == 1 and ("k_permute_direct" in placed[0]) <= (passes == 0), (n, ty, launched)
print("ok")
'''


@pytest.mark.parametrize("log4", [12, 13, 14])
def test_every_length_has_a_path(tmp_path, log4):
    lib = fake_hip.variant(tmp_path, "partition.hip", "CVLHIP_BLK_LOG4", log4)
    assert fake_hip.run(SCRIPT, tmp_path, lib=lib).startswith("ok")
