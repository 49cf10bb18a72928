"""Which way a permute with collisions goes, on the CPU: by source where few
sources aim at a long destination (below n_d / 32 of 2^21 or more), where
writing all of it would cost more than the launch that this saves."""
import fake_hip

SCRIPT = r'''
launched = []
fake, lib = load(lambda name, wgs, args: launched.append(name))
for n, n_d, few in ((100, 1 << 20, 0), (100, (1 << 21) - 1, 0), (100, 1 << 21, 1), ((1 << 16) - 1, 1 << 21, 1),
                    (1 << 16, 1 << 21, 0), (30_000, 3_000_000, 1), (90_000, 4_000_000, 1), (1 << 21, 1 << 22, 0)):
    for ty in "zd":
        launched.clear()
        getattr(lib, f"dpe_pu{ty}")(1 << 40, 1 << 41, 1 << 42, 1 << 43, n, n_d, 1 << 44)
        by_source, by_dest = (any(k in x for x in launched) for k in ("k_scatter_won", "k_place_won"))
        assert by_source == bool(few) and by_dest != by_source, (n, n_d, launched)
print("ok")
'''


def test_few_sources_of_long_destinations_go_by_source(tmp_path):
    assert fake_hip.run(SCRIPT, tmp_path).startswith("ok")
