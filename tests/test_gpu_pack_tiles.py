"""Packs whose tiles are counted first: one look-back tile (32768 ints, 16384
doubles) and the first length above it, the ends of the counted tiles (4096
ints, 2048 doubles), the last counted length (2^24) and the first after it;
flags of any non-zero value, none, all or a few; unaligned vectors."""
import pytest

pytestmark = pytest.mark.gpu

SIZES = [16385, 32768, 32769, 10 * 4096, 10 * 4096 + 1, 11 * 4096 - 1, 1_000_003, 1 << 24, (1 << 24) + 1]


@pytest.fixture(scope="module")
def cv():
    from neslgpu_amd.cvl import Cvl
    return Cvl()


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("ty", ["z", "d"])
def test_pack_tiles(cv, ty, n):
    import torch
    L, dev = cv.lib, cv.device
    dt = torch.float64 if ty == "d" else torch.int32
    g = torch.Generator(device=dev)
    g.manual_seed(n)
    s0 = torch.arange(n, device=dev).to(dt) + 1
    print("pack", ty, n, flush=True)
    for share in (0.0, 0.02, 0.5, 1.0):
        f0 = torch.where(torch.rand(n, generator=g, device=dev) < share,
                         torch.randint(1, 1 << 30, (n,), generator=g, device=dev, dtype=torch.int32), 0)
        for shift in (0, 1):
            s = torch.empty(n + shift, dtype=dt, device=dev)[shift:]
            f = torch.empty(n + shift, dtype=torch.int32, device=dev)[shift:]
            s.copy_(s0)
            f.copy_(f0)
            want = s[f != 0]
            k = L.pk1_luv(f, n, cv.scratch(L.pk1_luv_scratch(n)))
            assert k == want.numel()
            d = torch.full((k + 1,), -7, dtype=dt, device=dev)
            getattr(L, f"pk2_lu{ty}")(d, s, f, n, k, cv.scratch(getattr(L, f"pk2_lu{ty}_scratch")(n)))
            assert torch.equal(d[:k], want) and float(d[k]) == -7.0, (n, share, shift)
    assert L.cvlhip_check_device_errors() == 0
