"""The calls whose speed counts: CVL primitives and the short sequences of
them that a NESL program issues, through the Python binding of the C API.

Each family stands for work the VCODE programs and the benchmark do:

  reduce    a host-returning reduction (+_REDUCE, MAX_REDUCE): every
            MAKE_SEGDES and every IF over a vector waits for one
  scan      an unsegmented scan (+_SCAN, MAX_SCAN)
  segments  a segmented scan and a segmented reduction of the same values
            over uneven segments
  pack      PACK of a flat vector: count to the host, then compaction
  permute   PERMUTE by a random or a structured permutation
  rank      RANK of a key vector
  sort      RANK, then PERMUTE of the keys into order
  spmv      y = A x in CSR: BPERMUTE, * and +_REDUCE over the rows
  cross     elementwise arithmetic: quickhull's cross product and test for
            doubles, a hash and select for ints
  nest      MAKE_SEGDES of a lengths vector, then DIST and INDEX over it
  split     one level of nested quicksort: pivots, three compares and
            packs, and the pieces put back together by DPERMUTE

Every descriptor, scratch area and output vector is allocated once, as the
interpreter's arena keeps them; what a call builds (a descriptor from
lengths that the program has just computed) is built inside the pass.
"""
import math

import numpy as np
import torch

DEV = "cuda"
I32, I64, F64 = torch.int32, torch.int64, torch.float64

# work at both ends: a 1000-element reduction whose cost is one round trip,
# and 2^28-element vectors that fill the chip and its memory system
LISTED = [
    # the smallest call of a program: the total of a short lengths vector
    {"name": "reduce_small", "op": "reduce", "ty": "z", "fn": "add", "n": 1000},
    # a short sort, launches and round trips only
    {"name": "sort_small", "op": "sort", "ty": "z", "n": 5000, "up": True, "keys": "uniform"},
    # the plain scan at the benchmark's size
    {"name": "scan_int_large", "op": "scan", "ty": "z", "fn": "add", "n": 1 << 28},
    # the irregular float64 workload: heavy-tailed segments, as flattened
    # nested parallelism makes them
    {"name": "segments_f64_large", "op": "segments", "ty": "d", "scan": "add", "red": "max", "n": 1 << 26,
     "m": 51639, "lens": "zipf", "empties": False},
    # PACK of a long odd-sized vector, half the flags set
    {"name": "pack_int", "op": "pack", "ty": "z", "n": 100_000_007, "share": 0.5},
    # the random permutation of the benchmark
    {"name": "permute_large", "op": "permute", "ty": "z", "n": 1 << 28, "order": "random"},
    # the radix rank of the benchmark
    {"name": "rank_large", "op": "rank", "ty": "z", "n": 1 << 26, "up": True, "keys": "uniform"},
    # an ordinary sort of doubles, descending
    {"name": "sort_f64", "op": "sort", "ty": "d", "n": 3_000_001, "up": False, "keys": "uniform"},
    # the sparse product of the benchmark: 2^22 power-law rows, 2^26 nonzeros
    {"name": "spmv_large", "op": "spmv", "n": 1 << 26, "m": 1 << 22, "cols": 1 << 22, "lens": "power",
     "empties": False},
    # quickhull's test of 2^24 points against lines
    {"name": "cross_f64", "op": "cross", "ty": "d", "n": 1 << 24},
    # a descriptor of a few hundred thousand short segments, and the two
    # calls that nearly always follow it
    {"name": "nest_mid", "op": "nest", "ty": "d", "n": 5_000_011, "m": 300_007, "lens": "geometric", "empties": True},
    # a level in the middle of a quicksort of 2^20 keys
    {"name": "split_mid", "op": "split", "n": 1 << 20, "m": 1 << 14, "lens": "geometric", "empties": False},
]


def listed():
    return [dict(c) for c in LISTED]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    """Another case of the families above: sizes log-uniform from a thousand
    elements to the listed largest, odd ones as often as they come."""
    op = rng.choice(["reduce", "scan", "segments", "segments", "pack", "permute", "rank", "sort", "spmv", "cross",
                     "nest", "split"])
    ty = rng.choice("zd")
    lens = rng.choice(["geometric", "zipf", "const"])
    empties = rng.random() < 0.4
    if op == "reduce":
        return {"op": op, "ty": ty, "fn": rng.choice(["add", "max", "min"]), "n": _log(rng, 1000, 1 << 27)}
    if op == "scan":
        return {"op": op, "ty": ty, "fn": rng.choice(["add", "max"]), "n": _log(rng, 1000, 1 << 27)}
    if op == "segments":
        n = _log(rng, 1000, 1 << 26)
        return {"op": op, "ty": ty, "scan": rng.choice(["add", "max"]), "red": rng.choice(["add", "max"]), "n": n,
                "m": _log(rng, 2, n // 4), "lens": lens, "empties": empties}
    if op == "pack":
        return {"op": op, "ty": ty, "n": _log(rng, 1000, 1 << 26), "share": rng.choice([0.05, 0.5, 0.9])}
    if op == "permute":
        return {"op": op, "ty": ty, "n": _log(rng, 1000, 1 << 26),
                "order": rng.choice(["random", "random", "transpose", "rotate"])}
    if op == "rank" or op == "sort":
        return {"op": op, "ty": ty, "n": _log(rng, 1000, 1 << (25 if ty == "z" else 23)),
                "up": rng.random() < 0.5, "keys": rng.choice(["uniform", "uniform", "small"])}
    if op == "spmv":
        n = _log(rng, 10000, 1 << 25)
        m = max(16, n // rng.choice([4, 16, 64]))
        return {"op": op, "n": n, "m": m, "cols": m, "lens": rng.choice(["power", "geometric"]), "empties": empties}
    if op == "cross":
        return {"op": op, "ty": ty, "n": _log(rng, 1000, 1 << 24)}
    n = _log(rng, 2000, 1 << 25 if op == "nest" else 1 << 22)
    m = _log(rng, 16, n // 4)
    if op == "nest":
        return {"op": op, "ty": ty, "n": n, "m": m, "lens": lens, "empties": empties}
    return {"op": op, "n": n, "m": m, "lens": lens, "empties": False}


# ------------------------------------------------------------------ inputs
def _gen(case, seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1_000_003 + salt * 7919 + int(case["n"])) & 0x7FFFFFFFFFFFFFFF)
    return g


def _ints(g, n, lo=-2 ** 31, hi=2 ** 31):
    return torch.randint(lo, hi, (n,), generator=g, device=DEV, dtype=I32)


def _doubles(g, n):
    """Uniform in [-1, 1), all 53 bits of the mantissa drawn."""
    return torch.rand(n, generator=g, device=DEV, dtype=F64).mul_(2.0).sub_(1.0)


def _values(g, n, ty):
    return _doubles(g, n) if ty == "d" else _ints(g, n)


def _lengths(case, g):
    """m segment lengths that sum to n: proportional to exponential
    ("geometric"), clipped power-law ("zipf", "power": the sparse rows) or
    equal weights, every segment with an element or, with empties, one in
    eight without."""
    n, m, kind = case["n"], case["m"], case["lens"]
    u = torch.rand(m, generator=g, device=DEV, dtype=F64).clamp_(min=1e-12)
    if kind == "geometric":
        w = -torch.log(u)
    elif kind == "zipf":
        w = u.pow(-2.0).clamp_(max=float(1 << 20))
    elif kind == "power":
        w = u.pow(-1.0 / 1.1).clamp_(max=float(1 << 14))
    else:
        w = torch.ones_like(u)
    live = torch.ones(m, device=DEV, dtype=torch.bool)
    if case["empties"]:
        live = torch.rand(m, generator=g, device=DEV) >= 0.125
        live[m // 2] = True
    k = int(live.sum())
    w = torch.where(live, w, torch.zeros_like(w))
    lens = torch.floor(w * ((n - k) / float(w.sum()) * (1.0 - 1e-9))).to(I64) + live.to(I64)
    left = n - int(lens.sum())                      # what the rounding left: spread over the live segments
    order = torch.nonzero(live).flatten()
    lens[order] += left // k
    lens[order[: left % k]] += 1
    assert int(lens.sum()) == n and int(lens.min()) >= 0
    return lens.to(I32)


def _permutation(case, g):
    n = case["n"]
    if case["order"] == "random":
        return torch.randperm(n, generator=g, device=DEV).to(I32)
    i = torch.arange(n, device=DEV, dtype=I64)
    if case["order"] == "rotate":
        by = int(torch.randint(0, n, (1,), generator=g, device=DEV))
        return ((i + by) % n).to(I32)
    cols = max(1, int(math.isqrt(n)))               # row-major to column-major, a ragged last row kept in place
    rows = n // cols
    p = torch.where(i < rows * cols, (i % cols) * rows + i // cols, i)
    return p.to(I32)


def _keys(case, g):
    n = case["n"]
    if case["keys"] == "small":
        k = _ints(g, n, 0, 1000)
        return k.to(F64) if case["ty"] == "d" else k
    return _values(g, n, case["ty"])


def _kept(case):
    return int(case["share"] * case["n"])


def _inputs(case, seed):
    op, n = case["op"], case["n"]
    g = _gen(case, seed, 1)
    if op in ("reduce", "scan"):
        return {"s": _values(g, n, case["ty"])}
    if op == "segments":
        return {"s": _values(g, n, case["ty"]), "lens": _lengths(case, g)}
    if op == "pack":
        f = torch.zeros(n, device=DEV, dtype=I32)       # a share of the flags, anywhere
        f[torch.randperm(n, generator=g, device=DEV)[:_kept(case)]] = 1
        return {"s": _values(g, n, case["ty"]), "f": f}
    if op == "permute":
        return {"s": _values(g, n, case["ty"]), "p": _permutation(case, g)}
    if op in ("rank", "sort"):
        return {"s": _keys(case, g)}
    if op == "spmv":
        return {"lens": _lengths(case, g), "cols": _ints(g, n, 0, case["cols"]), "vals": _doubles(g, n),
                "x": _doubles(g, case["cols"])}
    if op == "cross":
        if case["ty"] == "d":
            return {k: _doubles(g, n) for k in ("px", "py", "ax", "ay", "bx", "by")}
        return {"a": _ints(g, n), "b": _ints(g, n)}
    if op == "nest":
        m = case["m"]
        return {"lens": _lengths(case, g), "v": _values(g, m, case["ty"]), "start": _ints(g, m, 0, 1 << 20),
                "step": _ints(g, m, 1, 4)}
    return {"lens": _lengths(case, g), "s": _ints(g, n, 0, 2 ** 31 - 1)}


# ------------------------------------------------------------------ a program's state
class _State:
    pass


def prepare(case, seed):
    from neslgpu_amd.cvl import Cvl
    st = _State()
    st.case = case
    st.cv = cv = Cvl()
    L = st.L = cv.lib
    st.i = x = _inputs(case, seed)
    op, n, ty = case["op"], case["n"], case.get("ty", "z")
    dt = F64 if ty == "d" else I32
    units = [1]
    if op == "reduce":
        units.append(getattr(L, f"{case['fn']}_ru{ty}_scratch")(n))
    elif op == "scan":
        st.d = cv.empty(n, dt)
        units.append(getattr(L, f"{case['fn']}_su{ty}_scratch")(n))
    elif op == "segments":
        st.sd, st.d, st.r = cv.segd(x["lens"]), cv.empty(n, dt), cv.empty(case["m"], dt)
        units += [getattr(L, f"{case['scan']}_se{ty}_scratch")(n, case["m"]),
                  getattr(L, f"{case['red']}_re{ty}_scratch")(n, case["m"])]
    elif op == "pack":
        st.d = cv.empty(n, dt)
        units += [L.pk1_luv_scratch(n), getattr(L, f"pk2_lu{ty}_scratch")(n)]
    elif op == "permute":
        st.d = cv.empty(n, dt)
        units.append(getattr(L, f"smp_pu{ty}_scratch")(n))
    elif op in ("rank", "sort"):
        st.r = cv.empty(n, I32)
        units.append(getattr(L, f"rk{'u' if case['up'] else 'd'}_lu{ty}_scratch")(n))
        if op == "sort":
            st.d = cv.empty(n, dt)
            units.append(getattr(L, f"smp_pu{ty}_scratch")(n))
    elif op == "spmv":
        st.sd, st.t, st.y = cv.segd(x["lens"]), cv.empty(n, F64), cv.empty(case["m"], F64)
        units += [L.bck_pud_scratch(case["cols"], n), L.mul_wud_scratch(n), L.add_red_scratch(n, case["m"])]
    elif op == "cross":
        st.t = [cv.empty(n, dt) for _ in range(5)]
        st.f = cv.empty(n, I32)
    elif op == "nest":
        m = case["m"]
        st.sd = torch.zeros(L.siz_fos(n, m) * 2 + 64, dtype=I32, device=DEV)
        st.l2, st.d, st.ix = cv.empty(m, I32), cv.empty(n, dt), cv.empty(n, I32)
        units += [L.add_ruz_scratch(m), L.mke_fov_scratch(n, m)]
    else:
        m = case["m"]
        st.sd = cv.segd(x["lens"])
        st.m1, st.n1 = [cv.empty(m, I32) for _ in range(8)], [cv.empty(n, I32) for _ in range(5)]
        st.part = [torch.zeros(L.siz_fos(n, m) * 2 + 64, dtype=I32, device=DEV) for _ in range(3)]
        units += [L.add_suz_scratch(m), L.pk1_lev_scratch(n, m), L.add_ruz_scratch(m), L.mke_fov_scratch(n, m),
                  L.pk2_lez_scratch(n, m, n, m), L.dpe_puz_scratch(n, n)]
    st.scr = torch.empty(max(units) * 8 + 256, dtype=torch.uint8, device=DEV)
    return st


def run(st):
    return _RUN[st.case["op"]](st, st.L, st.i, st.scr, st.case, st.case["n"], st.case.get("ty", "z"))


def _reduce(st, L, x, scr, case, n, ty):
    r = getattr(L, f"{case['fn']}_ru{ty}")(x["s"], n, scr)
    return np.float64(r) if ty == "d" else r


def _scan(st, L, x, scr, case, n, ty):
    getattr(L, f"{case['fn']}_su{ty}")(st.d, x["s"], n, scr)
    return st.d


def _segments(st, L, x, scr, case, n, ty):
    getattr(L, f"{case['scan']}_se{ty}")(st.d, x["s"], st.sd, n, case["m"], scr)
    getattr(L, f"{case['red']}_re{ty}")(st.r, x["s"], st.sd, n, case["m"], scr)
    return st.d, st.r


def _pack(st, L, x, scr, case, n, ty):
    k = L.pk1_luv(x["f"], n, scr)
    getattr(L, f"pk2_lu{ty}")(st.d, x["s"], x["f"], n, k, scr)
    return k, st.d[:k]


def _permute(st, L, x, scr, case, n, ty):
    getattr(L, f"smp_pu{ty}")(st.d, x["s"], x["p"], n, scr)
    return st.d


def _rank(st, L, x, scr, case, n, ty):
    getattr(L, f"rk{'u' if case['up'] else 'd'}_lu{ty}")(st.r, x["s"], n, scr)
    return st.r


def _sort(st, L, x, scr, case, n, ty):
    _rank(st, L, x, scr, case, n, ty)
    getattr(L, f"smp_pu{ty}")(st.d, x["s"], st.r, n, scr)
    return st.r, st.d


def _spmv(st, L, x, scr, case, n, ty):
    L.bck_pud(st.t, x["x"], x["cols"], case["cols"], n, scr)
    L.mul_wud(st.t, st.t, x["vals"], n, scr)
    L.add_red(st.y, st.t, st.sd, n, case["m"], scr)
    return st.y, st.t


def _cross(st, L, x, scr, case, n, ty):
    t, f = st.t, st.f
    if ty == "d":                                   # (bx-ax)(py-ay) - (by-ay)(px-ax) > 0
        L.sub_wud(t[0], x["bx"], x["ax"], n, scr)
        L.sub_wud(t[1], x["py"], x["ay"], n, scr)
        L.sub_wud(t[2], x["by"], x["ay"], n, scr)
        L.sub_wud(t[3], x["px"], x["ax"], n, scr)
        L.mul_wud(t[0], t[0], t[1], n, scr)
        L.mul_wud(t[2], t[2], t[3], n, scr)
        L.sub_wud(t[0], t[0], t[2], n, scr)
        L.dis_vud(t[4], 0.0, n, scr)
        L.grt_wud(f, t[0], t[4], n, scr)
        return t[0], f
    L.mul_wuz(t[0], x["a"], x["b"], n, scr)         # a*b ^ (a+b), and the larger of it and a
    L.add_wuz(t[1], x["a"], x["b"], n, scr)
    L.xor_wuz(t[0], t[0], t[1], n, scr)
    L.les_wuz(f, t[0], x["a"], n, scr)
    L.sel_wuz(t[2], f, x["a"], t[0], n, scr)
    return t[2], f


def _nest(st, L, x, scr, case, n, ty):
    m = case["m"]
    total = L.add_ruz(x["lens"], m, scr)
    L.mke_fov(st.sd, x["lens"], total, m, scr)
    getattr(L, f"dis_ve{ty}")(st.d, x["v"], st.sd, total, m, scr)
    L.ind_lez(st.ix, x["start"], x["step"], st.sd, total, m, scr)
    L.len_fos(st.l2, st.sd, total, m, scr)
    return total, st.d, st.ix, st.l2


def _split(st, L, x, scr, case, n, ty):
    """less | equal | greater of every segment about its middle element."""
    m, a, b, s, sd = case["m"], st.m1, st.n1, x["s"], st.sd
    lens, half, offs, one, mid = a[:5]
    pivot, flag, kept_vals, at, out = b
    L.len_fos(lens, sd, n, m, scr)
    L.dis_vuz(half, 2, m, scr)
    L.div_wuz(half, lens, half, m, scr)
    L.ext_vez(mid, s, half, sd, n, m, scr)          # each segment's middle element
    L.dis_vez(pivot, mid, sd, n, m, scr)
    L.add_suz(offs, lens, m, scr)                   # where the pieces of each segment go
    L.dis_vuz(one, 1, m, scr)
    L.dis_vuz(out, 0, n, scr)
    for cnt, psd, test in zip(a[5:], st.part, (L.les_wuz, L.eql_wuz, L.grt_wuz)):
        test(flag, s, pivot, n, scr)
        L.pk1_lev(cnt, flag, sd, n, m, scr)
        kept = L.add_ruz(cnt, m, scr)
        L.mke_fov(psd, cnt, kept, m, scr)
        L.pk2_lez(kept_vals, s, flag, sd, n, m, psd, kept, m, scr)
        L.ind_lez(at, offs, one, psd, kept, m, scr)
        L.dpe_puz(out, kept_vals, at, out, kept, n, scr)    # over the vector itself, as the interpreter reuses it
        L.add_wuz(offs, offs, cnt, m, scr)
    return out, a[5], a[6], a[7]


_RUN = {"reduce": _reduce, "scan": _scan, "segments": _segments, "pack": _pack, "permute": _permute, "rank": _rank,
        "sort": _sort, "spmv": _spmv, "cross": _cross, "nest": _nest, "split": _split}


# ------------------------------------------------------------------ what a pass needs
def work(case):
    """Bytes of the calls of one pass, each call's inputs read once and its
    outputs written once (a descriptor counts as its m lengths), and the
    arithmetic operations on elements."""
    op, n, m = case["op"], case["n"], case.get("m", 0)
    w = 8 if case.get("ty") == "d" or op == "spmv" else 4
    if op == "reduce":
        return {"bytes": w * n, "flops": n}
    if op == "scan":
        return {"bytes": 2 * w * n, "flops": n}
    if op == "segments":
        return {"bytes": 3 * w * n + (8 + w) * m, "flops": 2 * n}
    if op == "pack":
        return {"bytes": (8 + w) * n + w * _kept(case), "flops": 2 * n}
    if op == "permute":
        return {"bytes": (2 * w + 4) * n, "flops": 0}
    if op == "rank":
        return {"bytes": (w + 4) * n, "flops": n}
    if op == "sort":
        return {"bytes": (w + 4) * n + (2 * w + 4) * n, "flops": n}
    if op == "spmv":
        gather, mul, red = 8 * case["cols"] + 4 * n + 8 * n, 24 * n, 8 * n + 12 * m
        return {"bytes": gather + mul + red, "flops": 2 * n}
    if op == "cross":
        return {"bytes": (7 * 24 + 8 + 20) * n if w == 8 else (4 * 12 + 16) * n, "flops": 8 * n if w == 8 else 5 * n}
    if op == "nest":
        return {"bytes": 4 * m + 4 * m + (4 + w) * m + w * n + 12 * m + 4 * n + 8 * m, "flops": 2 * n}
    setup = (8 + 4 + 12 + 12 + 8 + 8 + 4) * m + 8 * n                     # lengths, pivots, starts, the cleared result
    tests, counts, packs = 3 * 12 * n, 3 * (4 * n + 8 * m), 3 * 8 * n + 4 * n
    joins = 4 * n + 16 * n                                               # indices, then the pieces put in place
    return {"bytes": setup + tests + counts + packs + joins + 3 * (4 + 4 + 8 + 12) * m, "flops": 10 * n}


def tolerance(case):
    """Whole numbers, comparisons and moves are exact.  Double sums differ in
    the order of their additions only."""
    op, ty = case["op"], case.get("ty")
    if op == "spmv":
        return {"rel": 1e-15, "max": 1e-14}
    if ty == "d" and op == "reduce" and case["fn"] == "add":
        return {"rel": 1e-13}
    if ty == "d" and op in ("scan", "segments") and "add" in (case.get("fn"), case.get("scan"), case.get("red")):
        return {"rel": 1e-14, "max": 3e-14}
    return "exact"


# ------------------------------------------------------------------ plain 64-bit results
def _wrap(x):
    """int64 sums as the 32-bit ones that wrap."""
    return (((x + 2 ** 31) & 0xFFFFFFFF) - 2 ** 31).to(I32)


def _before(x):
    """Exclusive sums of a double vector, the leading 30 bits of each value
    added as integers, so that only the last bits round."""
    hi = torch.round(x * 2.0 ** 30)
    lo = x - hi * 2.0 ** -30
    h, l = hi.to(I64), lo
    return torch.cumsum(h, 0) - h, torch.cumsum(l, 0) - l


def _owner(lens):
    return torch.repeat_interleave(torch.arange(lens.numel(), device=DEV), lens.to(I64))


def _starts(lens):
    c = torch.cumsum(lens.to(I64), 0)
    return c - lens


def _seg_sum(x, lens):
    """Per-segment sums: of ints as they wrap, of doubles as above."""
    n = x.numel()
    at = _starts(lens)
    end = at + lens

    def total(v):
        c = torch.zeros(n + 1, device=DEV, dtype=v.dtype)
        torch.cumsum(v, 0, out=c[1:])
        return c[end] - c[at]

    if x.dtype == I32:
        return _wrap(total(x.to(I64)))
    hi = torch.round(x * 2.0 ** 30)
    return total(hi.to(I64)).to(F64) * 2.0 ** -30 + total(x - hi * 2.0 ** -30)


def _seg_scan_max(x, lens):
    """Exclusive running maxima from each segment's start: one running
    maximum over (segment number, order of the value) keys."""
    own = _owner(lens)
    uniq, inv = torch.unique(x, return_inverse=True)
    k = uniq.numel() + 1
    run = torch.cummax(own * k + inv, 0).values - own * k
    out = torch.empty_like(x)
    out[1:] = uniq[run[:-1].clamp_(max=k - 2)]
    heads = _starts(lens)[lens > 0]
    out[heads] = _lowest(x.dtype)
    return out


def _lowest(dtype):
    return -2 ** 31 if dtype == I32 else float(np.float32(-1.0e36))


def exact(case, seed):
    x, op, n, ty = _inputs(case, seed), case["op"], case["n"], case.get("ty", "z")
    if op == "reduce":
        s = x["s"]
        if case["fn"] == "add":
            if ty == "z":
                return int(_wrap(s.to(I64).sum()))
            return np.float64(_seg_sum(s, torch.tensor([n], device=DEV, dtype=I64))[0].item())
        v = (s.max() if case["fn"] == "max" else s.min()).item()
        return np.float64(v) if ty == "d" else v
    if op == "scan":
        s = x["s"]
        if case["fn"] == "add":
            if ty == "z":
                c = torch.cumsum(s, 0, dtype=I64)
                return _wrap(c - s)
            h, l = _before(s)
            return h.to(F64) * 2.0 ** -30 + l
        out = torch.empty_like(s)
        out[0] = _lowest(s.dtype)
        out[1:] = torch.cummax(s, 0).values[:-1]
        return out
    if op == "segments":
        s, lens = x["s"], x["lens"]
        if case["scan"] == "max":
            if n > 1 << 24:
                return None                          # the plain running maximum sorts all values first
            d = _seg_scan_max(s, lens)
        else:
            own, at = _owner(lens), _starts(lens).clamp(max=n - 1)
            if ty == "z":
                c = torch.cumsum(s, 0, dtype=I64) - s
                d = _wrap(c - c[at][own])
            else:
                h, l = _before(s)
                d = (h - h[at][own]).to(F64) * 2.0 ** -30 + (l - l[at][own])
        if case["red"] == "add":
            r = _seg_sum(s, lens)
        else:
            r = torch.full((lens.numel(),), _lowest(s.dtype), device=DEV, dtype=s.dtype)
            r.scatter_reduce_(0, _owner(lens), s, "amax", include_self=True)
        return d, r
    if op == "pack":
        kept = x["s"][x["f"] != 0]
        return int(kept.numel()), kept
    if op == "permute":
        d = torch.empty_like(x["s"])
        d[x["p"].to(I64)] = x["s"]
        return d
    if op in ("rank", "sort"):
        v, order = torch.sort(x["s"], stable=True, descending=not case["up"])
        r = torch.empty(n, device=DEV, dtype=I32)
        r[order] = torch.arange(n, device=DEV, dtype=I32)
        return r if op == "rank" else (r, v)
    if op == "spmv":
        t = x["x"][x["cols"].to(I64)] * x["vals"]
        return _seg_sum(t, x["lens"]), t
    if op == "cross":
        if ty == "d":
            c = (x["bx"] - x["ax"]) * (x["py"] - x["ay"]) - (x["by"] - x["ay"]) * (x["px"] - x["ax"])
            return c, (c > 0).to(I32)
        a, b = x["a"], x["b"]
        t = (a * b) ^ (a + b)
        f = t < a
        return torch.where(f, a, t), f.to(I32)
    lens = x["lens"]
    own, at = _owner(lens), _starts(lens)
    if op == "nest":
        k = torch.arange(n, device=DEV) - at[own]
        ix = _wrap(x["start"].to(I64)[own] + x["step"].to(I64)[own] * k)
        return n, x["v"][own], ix, lens
    s = x["s"]
    mid = s[at + torch.div(lens, 2, rounding_mode="floor")]
    pv = mid[own]
    side = (s >= pv).to(I64) + (s > pv).to(I64)      # 0 less, 1 equal, 2 greater
    order = torch.sort(own * 3 + side, stable=True).indices
    cnt = torch.bincount(own * 3 + side, minlength=3 * lens.numel()).view(-1, 3).to(I32)
    return s[order], cnt[:, 0].contiguous(), cnt[:, 1].contiguous(), cnt[:, 2].contiguous()
