"""Plain back-permutes at the ends of their tiles (1024 elements) and of the
rule for streamed ones (2^22), on aligned and unaligned vectors, over the
index vector itself, and with indices out of range (0 stored, error word
raised)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cv():
    from neslgpu_amd.cvl import Cvl
    return Cvl()


@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 50_001, (1 << 22) - 1, 1 << 22, (1 << 22) + 1025])
@pytest.mark.parametrize("ty", ["z", "d"])
def test_gather_tiles(cv, ty, n):
    import torch
    L, dev = cv.lib, cv.device
    dt = torch.float64 if ty == "d" else torch.int32
    g = torch.Generator(device=dev)
    g.manual_seed(n)
    n_s = 70_001
    s = torch.arange(n_s, device=dev).to(dt) * 2 + 1
    fn = getattr(L, f"bck_pu{ty}")
    print("gather", ty, n, flush=True)
    for shift in (0, 1):
        i = torch.empty(n + shift, dtype=torch.int32, device=dev)[shift:]
        i.copy_(torch.randint(0, n_s, (n,), generator=g, device=dev))
        d = torch.full((n + 1 + shift,), -7, dtype=dt, device=dev)[shift:]
        fn(d, s, i, n_s, n, None)
        want = s[i.long()]
        assert torch.equal(d[:n], want) and float(d[n]) == -7.0, (n, shift)
        assert L.cvlhip_check_device_errors() == 0
        bad = i.clone() if shift == 0 else torch.cat([i[:1], i])[1:]
        bad[n // 2], bad[0] = n_s, -1
        fn(d, s, bad, n_s, n, None)
        want[n // 2] = 0
        want[0] = 0
        assert torch.equal(d[:n], want) and float(d[n]) == -7.0, (n, shift, "range")
        assert L.cvlhip_check_device_errors() != 0
        if ty == "z":
            want = s[i.long()]
            fn(i, s, i, n_s, n, None)
            assert torch.equal(i, want), (n, shift, "in place")
