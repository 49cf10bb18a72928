"""Elementwise calls at the ends of their tiles (one 16-byte vector per lane
below 2^21 elements, two above: 512 to 2048 elements per workgroup), on
aligned and unaligned operands and over their own inputs, against torch."""
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 511, 512, 513, 1023, 1024, 1025, 100_003, (1 << 21) - 1, 1 << 21, (1 << 21) + 1, (1 << 21) + 2049]


@pytest.fixture(scope="module")
def cv():
    from neslgpu_amd.cvl import Cvl
    return Cvl()


def vec(cv, x, shift):
    import torch
    t = torch.empty(x.numel() + shift, dtype=x.dtype, device=cv.device)[shift:]
    t.copy_(x)
    return t


@pytest.mark.parametrize("n", SIZES)
def test_elementwise_tiles(cv, n):
    import torch
    L, dev = cv.lib, cv.device
    g = torch.Generator(device=dev)
    g.manual_seed(n)
    za, zb = (torch.randint(-2 ** 31, 2 ** 31, (n,), generator=g, device=dev, dtype=torch.int32) for _ in range(2))
    da, db = (torch.rand(n, generator=g, device=dev, dtype=torch.float64) - 0.5 for _ in range(2))
    fl = torch.randint(0, 3, (n,), generator=g, device=dev, dtype=torch.int32)
    i32, f64 = torch.int32, torch.float64
    cases = [("add_wuz", (za, zb), za + zb), ("les_wuz", (za, zb), (za < zb).to(i32)), ("sub_wud", (da, db), da - db),
             ("grt_wud", (da, db), (da > db).to(i32)), ("not_wuz", (za,), ~za), ("sqt_wud", (da.abs(),), da.abs().sqrt()),
             ("int_wud", (da * 100,), (da * 100).to(i32)), ("dbl_wuz", (za,), za.to(f64)),
             ("boo_wuz", (fl,), (fl != 0).to(i32)), ("sel_wuz", (fl, za, zb), torch.where(fl != 0, za, zb)),
             ("sel_wud", (fl, da, db), torch.where(fl != 0, da, db))]
    print("elementwise", n, flush=True)
    for name, args, want in cases:
        for shift in (0, 1):
            ins = [vec(cv, a, shift) for a in args]
            d = torch.full((n + 1 + shift,), 7, dtype=want.dtype, device=dev)[shift:]
            getattr(L, name)(d, *ins, n, None)
            assert torch.equal(d[:n], want), (name, n, shift)
            assert float(d[n]) == 7.0, (name, n, shift)
            if name in ("add_wuz", "sub_wud", "not_wuz"):           # over an input
                getattr(L, name)(ins[-1], *ins, n, None)
                assert torch.equal(ins[-1], want), (name, n, shift, "in place")
    for shift in (0, 1):
        d = torch.zeros(n + 1 + shift, dtype=i32, device=dev)[shift:]
        L.ind_luz(d, -5, 3, n, None)
        assert torch.equal(d[:n], torch.arange(n, device=dev, dtype=i32) * 3 - 5) and int(d[n]) == 0
        e = torch.zeros(n + 1 + shift, dtype=f64, device=dev)[shift:]
        L.dis_vud(e, 0.25, n, None)
        assert bool((e[:n] == 0.25).all()) and float(e[n]) == 0.0
    assert L.cvlhip_check_device_errors() == 0
