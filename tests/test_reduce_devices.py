"""The memory in which the blocks of a host-returning reduction meet belongs
to the device of the call, on the CPU: reductions of several blocks on two
devices in turn, each launched with memory of its own device, which stays the
same from call to call; where there is none (more devices than the library
keeps it for), the second launch posts the result."""
import fake_hip

SCRIPT = r'''
import ctypes as C
calls = []

def on_launch(name, wgs, args):
    # (in, n, ..., share, mailbox, number, error word); k_reduce has one argument more before them
    at = {"k_reduce_strided": 5, "k_reduceI": 6}
    for k, i in at.items():
        if k in name:
            share = word(args, i)
            calls.append((name, wgs, share))
            if share:
                Post.to(word(args, i + 1), word(args, i + 2), 7)
            return
    if "k_reduce_finish" in name:
        calls.append((name, wgs, None))
        Post.to(word(args, 3), word(args, 4), 9)

fake, lib = load(on_launch)
n = 3_000_000
seen = {}
for device in (0, 1, 0, 1, 5, 0):
    fake.fake_set_device(device)
    for f in (lib.add_ruz, lib.max_rud, lib.add_rud, lib.pk1_luv):
        calls.clear()
        assert int(f(1 << 45, n, 1 << 46)) in (0, 7), f      # (a double of the bits 7 is 0.0 in whole numbers)
        assert len(calls) == 1 and calls[0][1] > 1, calls
        share = calls[0][2]
        assert fake.fake_device_of(share) == device, (device, f, fake.fake_device_of(share))
        assert seen.setdefault(device, share) == share
assert len(set(seen.values())) == 3
fake.fake_set_device(64)
calls.clear()
assert lib.add_ruz(1 << 45, n, 1 << 46) == 9
assert [c[2] for c in calls] == [0, None], calls
print("ok")
'''


def test_the_blocks_meet_in_their_own_devices_memory(tmp_path):
    assert fake_hip.run(SCRIPT, tmp_path).startswith("ok")
