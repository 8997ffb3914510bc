"""What the framework is timed on: the work its users have it do, through the
public entry points (the C ABI as the package binds it, and the package's
deep scan), on inputs resident on the GPU where the path keeps them there.

Polynomials over GF(2) are int64 tensors of little-endian words; every output
is whole words, so two builds agree bit for bit or not at all.
"""
import ctypes as C
import math
import random

import numpy as np
import torch

import mersenne_trinomial_amd as M
from mersenne_trinomial_amd import device
from mersenne_trinomial_amd._capi import check, lib

R_FULL = 136279841
# the trinomial degrees the tests, the benchmark and the serving mix run
DEGREES = (4423, 9689, 132049, 756839, 3021377, R_FULL)


def listed():
    return [
        # one residue's Frobenius chain at the smallest degree a search runs:
        # a handful of tiny launches, so launch latency counts
        {"name": "chain_one_132049", "kind": "chain", "r": 132049, "n": 1, "steps": 40,
         "uneven": False, "mixed": False},
        # survivors at frontiers of their own, several trinomial degrees in
        # one batch (the shape of a serving mix)
        {"name": "chain_mixed_48", "kind": "chain", "r": 3021377, "n": 48, "steps": 24,
         "uneven": True, "mixed": True},
        # the batched chain of the full-size search, the benchmark's step
        {"name": "chain_full_64", "kind": "chain", "r": R_FULL, "n": 64, "steps": 64,
         "uneven": False, "mixed": False},
        # a modular product of the smallest search: an interval product's step
        {"name": "mulmod_132049", "kind": "mul", "abits": 132049, "bbits": 132049, "r": 132049},
        # a plain product of two different, ragged sizes
        {"name": "mul_3021377x1000003", "kind": "mul", "abits": 3021377, "bbits": 1000003, "r": 0},
        # the full-size modular product
        {"name": "mulmod_full", "kind": "mul", "abits": R_FULL, "bbits": R_FULL, "r": R_FULL},
        # many products of different sizes, each folded (the benchmark's
        # product batch)
        {"name": "mul_batch_64", "kind": "batch", "n": 64, "lo": 16.0, "hi": 27.0, "r": R_FULL},
        # transforms used by themselves, forward and inverse
        {"name": "transform_20", "kind": "fft", "m": 20},
        # the deep scan's unit of device work: a block of m degrees of a
        # cohort (Horner product, interval product, m squarings of the table)
        {"name": "block_full_4x32", "kind": "block", "r": R_FULL, "n": 4, "m": 32},
        # coarse sieves: a whole small search, and the whole full-size one
        {"name": "sieve_132049_d20", "kind": "sieve", "r": 132049, "depth": 20, "smax": 66024},
        {"name": "sieve_full_d32", "kind": "sieve", "r": R_FULL, "depth": 32, "smax": 68139920},
        # a deep scan from survivors to certificate rows: device blocks,
        # interval gcds on host threads with device products, resolution
        {"name": "scan_756839", "kind": "scan", "r": 756839, "n": 8, "k0": 20, "maxd": 512},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["chain", "chain", "mul", "mul", "mul", "batch", "fft", "block", "sieve",
                       "scan"])
    if kind == "chain":
        n = _log(rng, 1, 64)
        r = _log(rng, 1001, R_FULL if n > 4 else 4 * R_FULL // 3)
        return {"kind": kind, "r": r, "n": n, "steps": rng.randint(1, 64),
                "uneven": bool(n > 1 and rng.random() < 0.5),
                "mixed": bool(n > 1 and rng.random() < 0.3)}
    if kind == "mul":
        a = _log(rng, 1000, R_FULL)
        b = a if rng.random() < 0.5 else _log(rng, max(1000, a // 64), a)
        fold = rng.random() < 0.6
        return {"kind": kind, "abits": a, "bbits": b,
                "r": rng.choice([a, max(a, (a + b + 1) // 2 + rng.randint(0, 200))]) if fold else 0}
    if kind == "batch":
        lo = rng.uniform(10.0, 20.0)
        return {"kind": kind, "n": _log(rng, 2, 64), "lo": lo,
                "hi": rng.uniform(lo, 26.5), "r": R_FULL}
    if kind == "fft":
        return {"kind": kind, "m": rng.randint(8, 24)}
    if kind == "block":
        r = _log(rng, 100003, R_FULL)
        m = rng.choice([8, 16, 24, 32])
        return {"kind": kind, "r": r, "n": max(1, min(64, int(4e9 / (m * r)) or 1, rng.randint(1, 64))),
                "m": m}
    if kind == "sieve":
        r = rng.choice(DEGREES)
        d = rng.randint(12, 31)
        return {"kind": kind, "r": r, "depth": d, "smax": _log(rng, 1000, 50 * r // 100 - 1)}
    r = rng.choice(DEGREES[2:4])
    return {"kind": "scan", "r": r, "n": _log(rng, 2, 8), "k0": rng.randint(16, 22),
            "maxd": _log(rng, 128, 512)}


# ------------------------------------------------------------------ inputs
def _words(bits):
    return (bits + 63) >> 6


def _random_bits(gen, bits):
    """`bits` uniform random bits, zero above, in an int64 tensor."""
    w = _words(bits)
    t = torch.randint(-2**63, 2**63 - 1, (w,), dtype=torch.int64, device="cuda", generator=gen)
    if bits & 63:
        t[-1] &= (1 << (bits & 63)) - 1
    return t


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _ptrs(tensors):
    return (C.c_void_p * len(tensors))(*[t.data_ptr() for t in tensors])


def _u64s(v):
    return (C.c_uint64 * len(v))(*[int(x) for x in v])


def _bytes(n):
    return torch.empty((int(n) + 7) // 8 + 1, dtype=torch.int64, device="cuda")


def _s_values(rng, r, n):
    return [rng.randint(1, (r - 1) // 2) for _ in range(n)]


def _chain_shape(case):
    """degree and step count of each residue (the case's, whatever the seed)"""
    rng = random.Random(case["r"] + case["n"])
    n = case["n"]
    rs = [case["r"]] * n
    if case["mixed"]:
        small = [d for d in DEGREES if d <= case["r"]] or [case["r"]]
        rs = [rng.choice(small) for _ in range(n)]
    steps = [rng.randint(1, case["steps"]) if case["uneven"] else case["steps"] for _ in range(n)]
    return rs, steps


def _batch_shape(case):
    """bit lengths 2^lo..2^hi of each pair (the case's, whatever the seed)"""
    rng = random.Random(case["n"])
    top = min(case["r"], 1 << 27)
    ab = [min(top, int(2 ** rng.uniform(case["lo"], case["hi"]))) for _ in range(case["n"])]
    bb = [min(top, int(2 ** rng.uniform(case["lo"], case["hi"]))) for _ in range(case["n"])]
    return ab, bb


def prepare(case, seed):
    device.init()
    kind, gen, rng = case["kind"], _gen(seed), random.Random(seed + 1)
    st = {"kind": kind, "case": dict(case)}
    if kind == "chain":
        rs, steps = _chain_shape(case)
        ss = [rng.randint(1, (r - 1) // 2) for r in rs]
        x = [_random_bits(gen, r) for r in rs]
        st.update(x=x, tmp=[torch.empty_like(t) for t in x], rs=rs, ss=ss, steps=steps)
        if case["n"] > 1:
            st.update(px=_ptrs(x), pt=_ptrs(st["tmp"]), ar=_u64s(rs), as_=_u64s(ss),
                      ak=_u64s(steps))
    elif kind == "mul":
        a, b, r = case["abits"], case["bbits"], case["r"]
        st.update(a=_random_bits(gen, a), b=_random_bits(gen, b),
                  s=rng.randint(1, (r - 1) // 2) if r else 0,
                  out=torch.empty(_words(r) if r else lib.gf2t_mul_out_words(a, b),
                                  dtype=torch.int64, device="cuda"),
                  work=_bytes(lib.gf2t_mul_workspace_bytes(a, b)))
    elif kind == "batch":
        ab, bb = _batch_shape(case)
        ss = _s_values(rng, case["r"], case["n"])
        nw, n = _words(case["r"]), case["n"]
        a, b = [_random_bits(gen, k) for k in ab], [_random_bits(gen, k) for k in bb]
        out = torch.empty((n, nw), dtype=torch.int64, device="cuda")
        aa, bbv = _u64s(ab), _u64s(bb)
        st.update(a=a, b=b, out=out, pa=_ptrs(a), pb=_ptrs(b), po=_ptrs(list(out)), aa=aa, bb=bbv,
                  as_=_u64s(ss), work=_bytes(lib.gf2t_mulmod_batch_workspace_bytes(n, aa, bbv)))
    elif kind == "fft":
        F = M.DevFFT()
        F.init(case["m"])
        st.update(F=F, f=_random_bits(gen, 64 << case["m"]), g=_random_bits(gen, 64 << case["m"]))
        st.update(ff=torch.empty_like(st["f"]), gg=torch.empty_like(st["g"]))
    elif kind == "block":
        r, n, m = case["r"], case["n"], case["m"]
        nw = _words(r)
        pitch = (nw + 31) & ~31
        tab = torch.zeros((n * m, pitch), dtype=torch.int64, device="cuda")
        for i in range(n * m):
            tab[i, :nw] = _random_bits(gen, r)
        acc = torch.zeros((n, pitch), dtype=torch.int64, device="cuda")
        for i in range(n):
            acc[i, :nw] = _random_bits(gen, r)
        ss = _s_values(rng, r, n)
        plan = C.c_void_p()
        check(lib.gf2t_sq2_slab_plan_create(r, _u64s(ss), n, C.byref(plan)))
        st.update(tab=tab, alt=torch.zeros_like(tab), acc=acc, c=torch.zeros_like(acc), nw=nw,
                  pitch=pitch, plan=_Plan(plan), ds=torch.tensor(ss, dtype=torch.int64, device="cuda"),
                  work=_bytes(lib.gf2t_mulmod_slab_workspace_bytes(r, n)))
    elif kind == "sieve":
        # the image of an earlier run that resolved one s in sixteen by x^2+x+1
        # (the minimum a continued sieve starts from), and the working copy
        hit = torch.rand(case["smax"] + 1, device="cuda", generator=gen) < 1 / 16
        st["image"] = torch.where(hit, (2 << 48) | 7, -1)
        st["best"] = torch.empty_like(st["image"])
    else:
        r, k0 = case["r"], case["k0"]
        smax = min((r - 1) // 2, 20000)
        best = torch.full((smax + 1,), -1, dtype=torch.int64, device="cuda")
        check(lib.gf2t_sieve(r, 2, k0, smax, best.data_ptr(), None))
        left = torch.nonzero(best[1:] == -1).flatten().cpu().numpy() + 1
        pick = np.random.default_rng(seed).choice(left, size=min(case["n"], left.size), replace=False)
        st["svals"] = np.sort(pick).astype(np.uint64)
    return st


class _Plan:
    def __init__(self, h):
        self.h = h

    def __del__(self):
        torch.cuda.synchronize()
        lib.gf2t_sq2_slab_plan_destroy(self.h)


# ---------------------------------------------------------------- one pass
def run(st):
    kind, case = st["kind"], st["case"]
    if kind == "chain":
        if case["n"] == 1:
            check(lib.gf2t_square_fold_steps(st["x"][0].data_ptr(), st["tmp"][0].data_ptr(),
                                             st["rs"][0], st["ss"][0], st["steps"][0], None))
        else:
            check(lib.gf2t_square_fold_batch(st["px"], st["pt"], st["ar"], st["as_"], st["ak"],
                                             case["n"], None))
        return st["x"]
    if kind == "mul":
        a, b, r = case["abits"], case["bbits"], case["r"]
        if r:
            check(lib.gf2t_mulmod(st["a"].data_ptr(), a, st["b"].data_ptr(), b, r, st["s"],
                                  st["out"].data_ptr(), st["work"].data_ptr(), None))
        else:
            check(lib.gf2t_mul(st["a"].data_ptr(), a, st["b"].data_ptr(), b, st["out"].data_ptr(),
                               st["work"].data_ptr(), None))
        return st["out"]
    if kind == "batch":
        check(lib.gf2t_mulmod_batch(case["n"], st["pa"], st["aa"], st["pb"], st["bb"], case["r"],
                                    st["as_"], st["po"], st["work"].data_ptr(), None))
        return st["out"]
    if kind == "fft":
        st["ff"].copy_(st["f"])
        st["F"].fwd(st["ff"].data_ptr())
        st["gg"].copy_(st["g"])
        st["F"].inv(st["gg"].data_ptr())
        return [st["ff"], st["gg"]]
    if kind == "block":
        r, n, m, pitch, ds = case["r"], case["n"], case["m"], st["pitch"], st["ds"].data_ptr()
        cur, oth, acc, c = st["tab"], st["alt"], st["acc"].data_ptr(), st["c"].data_ptr()
        check(lib.gf2t_horner_slab(cur.data_ptr(), pitch, m, r, ds, c, pitch, n, None))
        check(lib.gf2t_mulmod_slab(acc, pitch, c, pitch, 0, r, ds, acc, pitch, n,
                                   st["work"].data_ptr(), None))
        for _ in range(m // 2):
            check(lib.gf2t_square2_fold_slab_p(st["plan"].h, cur.data_ptr(), oth.data_ptr(), pitch,
                                               n * m, m, None))
            cur, oth = oth, cur
        st["tab"], st["alt"] = cur, oth
        return [st["acc"][:, :st["nw"]], cur[:, :st["nw"]]]
    if kind == "sieve":
        st["best"].copy_(st["image"])
        check(lib.gf2t_sieve(case["r"], 2, case["depth"], case["smax"], st["best"].data_ptr(), None))
        return st["best"]
    rows = M.scan(case["r"], st["svals"], case["k0"], maxd=case["maxd"])
    # the certificate lines' fields; a factor's mask as its hex digits' bytes
    masks = np.zeros((len(rows), case["maxd"] // 4 + 1), dtype=np.uint8)
    for k, x in enumerate(rows):
        masks[k, :len(x.hex)] = np.frombuffer(x.hex.encode(), dtype=np.uint8)
    return [np.array([[x.s, x.kind, x.d, x.rlo, x.rhi, len(x.hex)] for x in rows], dtype=np.int64),
            masks]


def work(case):
    """Bytes: inputs read once, outputs written once.  flops: 32-bit integer
    operations on words that the arithmetic itself takes (one interleave of 21
    per 64 bits squared; a transform's GF(2^64) additions and products at one
    operation each; a class's table lookup)."""
    kind = case["kind"]
    if kind == "chain":
        words = case["n"] * _words(case["r"])
        return {"bytes": 16 * words, "flops": 21 * words * case["steps"]}
    if kind == "mul":
        a, b, r = case["abits"], case["bbits"], case["r"]
        return {"bytes": (a + b + (r or a + b)) // 8, "flops": _product_ops(a, b)}
    if kind == "batch":
        ab, bb = _batch_shape(case)
        return {"bytes": sum(a + b + case["r"] for a, b in zip(ab, bb)) // 8,
                "flops": sum(_product_ops(a, b) for a, b in zip(ab, bb))}
    if kind == "fft":
        return {"bytes": 32 << case["m"], "flops": 3 * case["m"] << case["m"]}
    if kind == "block":
        words = case["n"] * _words(case["r"])
        return {"bytes": words * (16 * case["m"] + 16),
                "flops": 21 * words * case["m"] * (case["m"] & ~1) + case["n"] * _product_ops(case["r"], case["r"])}
    if kind == "sieve":
        return {"bytes": 8 * (case["smax"] + 1), "flops": 2 << case["depth"]}
    words = case["n"] * _words(case["r"])
    return {"bytes": 16 * words, "flops": 21 * words * case["maxd"]}


def _product_ops(a, b):
    n = (a + b) / 32
    return int(3 * 1.5 * n * max(1.0, math.log2(n)))


# ------------------------------------------------------------------- exact
def _bits(t):
    return np.unpackbits(np.ascontiguousarray(t.cpu().numpy()).view(np.uint8), bitorder="little")


def _pack(bits, words):
    full = np.zeros(64 * words, dtype=np.uint8)
    full[:min(bits.size, full.size)] = bits[:full.size]
    return torch.from_numpy(np.packbits(full, bitorder="little").view(np.int64).copy())


def _fold(p, r, s):
    """reduce a 0/1 coefficient array of at most 2r - 1 entries mod x^r + x^s + 1"""
    p = np.concatenate([p, np.zeros(max(0, 2 * r - p.size), dtype=np.uint8)])
    for _ in range(2):
        hi = p[r:].copy()
        p[r:] = 0
        p[:hi.size] ^= hi
        p[s:s + hi.size] ^= hi
    return p[:r]


def exact(case, seed):
    """The residues and products in plain numpy for sizes where that is quick
    (squaring as bit spread and fold, a product as an integer convolution in
    float64, exact at these lengths); the other paths have whole-number
    outputs that only a second implementation could give."""
    st = prepare(case, seed)
    if case["kind"] == "chain" and sum(r * k for r, k in zip(st["rs"], st["steps"])) < 3e8:
        out = []
        for x, r, s, k in zip(st["x"], st["rs"], st["ss"], st["steps"]):
            v = _bits(x)[:r]
            for _ in range(k):
                sq = np.zeros(2 * r, dtype=np.uint8)
                sq[::2] = v
                v = _fold(sq, r, s)
            out.append(_pack(v, _words(r)))
        return out
    if case["kind"] == "mul" and case["abits"] + case["bbits"] < 1 << 23:
        a, b, r = case["abits"], case["bbits"], case["r"]
        n = 1 << (a + b).bit_length()
        f = np.fft.rfft(_bits(st["a"])[:a].astype(np.float64), n)
        g = np.fft.rfft(_bits(st["b"])[:b].astype(np.float64), n)
        p = (np.rint(np.fft.irfft(f * g, n)).astype(np.int64) & 1).astype(np.uint8)[:a + b - 1]
        if r:
            return _pack(_fold(p, r, st["s"]), _words(r))
        return _pack(p, int(lib.gf2t_mul_out_words(a, b)))
    return None
