"""The work whose speed is measured: two-operand contractions and products, and
the fused linear-attention chain, through the package's public entry points.

Families (``family`` of a case) and what each stands for:

  matmul      one-shot ``einsum()`` of two matrices, from latency-sized to
              8192^3, both dtypes, every layout of the operands, odd extents;
  batched     a kept runner of a batched contraction whose operands are stored
              transposed (``bji,bjk->bik`` and its siblings);
  attention   multi-head scores and values of a prefill step;
  decode      the scores and values of one new token per sequence against a
              key / value cache;
  matvec      a matrix against a vector, a dot product, rows against rows;
  multi_axis  contractions over several axes whose order differs between the
              operands, projections to and from heads;
  chunk       the four contractions of a chunked gated-delta-rule stage, eager;
  product     Hadamard and broadcast products (decay masks, norm scales,
              rotary tables);
  linattn     ``linear_attention(q, k, v, m)``.

Inputs are drawn on the GPU from the seed.  Runners are built in ``prepare``
as a program that calls an equation repeatedly keeps them; ``matmul`` cases
call ``einsum`` itself, whose runner cache does that.
"""
import os
import sys
import tempfile
from math import prod

import torch

# The package lives in a folder of the repository whose root is the working
# directory here.
sys.path.insert(0, os.path.abspath("pto-einsum_amd"))

# Generated per-shape libraries go to a folder of this process's own (the
# default, ./build, needs a writable working directory).
_BUILD = tempfile.TemporaryDirectory(prefix="pto_einsum_")
os.environ["EINSUM_BUILD_DIR"] = _BUILD.name

from pto_einsum import EinsumBuilder, einsum, linear_attention  # noqa: E402

DEV = "cuda"
DTYPES = {"float32": torch.float32, "float16": torch.float16}


def _dims(eq, text):
    """Extents by axis letter from a case's "i=256 j=256" text."""
    d = {k: int(v) for k, v in (x.split("=") for x in text.split())}
    assert set(d) == set(eq) - set(",->"), (eq, text)
    return d


def _eqs(case):
    """The (equation, extents) pairs that a pass of an einsum case computes."""
    if case["family"] == "chunk":
        b, h, n, d = case["b"], case["h"], case["n"], case["d"]
        return [(eq, dict(zip("bihjdve", (b, n, h, n, d, n, d)))) for eq in CHUNK_EQS]
    if case["family"] == "decode":
        b, h, t, d = case["b"], case["h"], case["t"], case["d"]
        return [(eq, dict(b=b, h=h, t=t, d=d)) for eq in DECODE_EQS]
    return [(case["eq"], _dims(case["eq"], case["dims"]))]


# kkt, wy_fast, the state's outer product and the state's read-out of a
# chunked gated-delta-rule stage (n tokens a chunk, d channels a head).
CHUNK_EQS = ("bihd,bjhd->bihj", "bihj,bjhd->bihd", "bvhd,bvhe->bhde", "bvhd,bhde->bvhe")
DECODE_EQS = ("bhd,bthd->bht", "bht,bthd->bhd")


def _split(eq):
    ins, out = eq.split("->")
    a, b = ins.split(",")
    return a, b, out


def listed():
    return [
        # The smallest call: one matrix product of the size at which the
        # launch and the host's work for it outweigh the arithmetic.
        dict(name="matmul_small", family="matmul", eq="ij,jk->ik", dims="i=256 j=256 k=256", dtype="float32"),
        # A product whose extents are what data gives (none a multiple of
        # eight), so rows start unaligned.
        dict(name="matmul_odd", family="matmul", eq="ij,jk->ik", dims="i=2001 j=1537 k=3003", dtype="float16"),
        # The largest product: a square one of float16 matrices, the second
        # stored by rows of its columns, as a weight is.
        dict(name="matmul_large", family="matmul", eq="ij,kj->ik", dims="i=8192 j=8192 k=8192", dtype="float16"),
        # Batched and transposed, extents no multiples of 16.
        dict(name="batched_transposed", family="batched", eq="bji,bjk->bik", dims="b=16 j=777 i=1000 k=1536",
             dtype="float32"),
        # Prefill attention scores; the output is by far the largest tensor.
        dict(name="attention_scores", family="attention", eq="bshd,bthd->bsht", dims="b=4 s=2048 t=2048 h=32 d=128",
             dtype="float16"),
        # One decoded token: 16 sequences, 32 heads, 2048 cached positions.
        dict(name="decode", family="decode", b=16, h=32, t=2048, d=128, dtype="float16"),
        # A matrix times a vector.
        dict(name="matvec", family="matvec", eq="ij,j->i", dims="i=8192 j=4096", dtype="float32"),
        # Two contracted axes that the operands store in opposite order.
        dict(name="multi_axis", family="multi_axis", eq="ikj,jlk->il", dims="i=768 k=48 j=64 l=1000", dtype="float32"),
        # A gated-delta-rule stage: 64 chunks of 128 tokens, 16 heads.
        dict(name="chunk_stage", family="chunk", b=64, h=16, n=128, d=128, dtype="float32"),
        # The decay mask of linear attention applied to its scores.
        dict(name="hadamard", family="product", eq="ts,ts->ts", dims="t=4096 s=4096", dtype="float32"),
        # Rotary table times activations.
        dict(name="broadcast", family="product", eq="bshd,sd->bshd", dims="b=2 s=4096 h=32 d=128", dtype="float16"),
        # The fused chain over 4096 positions.
        dict(name="linear_attention", family="linattn", t=4096, s=4096, n=128, p=128, dtype="float16", precise=False),
    ]


# ------------------------------------------------------------------ drawing --

def _size(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi]: as it falls, or rounded
    to a multiple of 8 or 64 as configured sizes are."""
    n = int(round(lo * (hi / lo) ** rng.random()))
    step = rng.choice([1, 1, 8, 64])
    return min(hi, max(lo, n // step * step))


def _text(eq, d):
    return " ".join("%s=%d" % (c, d[c]) for c in dict.fromkeys(c for c in eq if c.isalpha()))


def draw(rng):
    while True:
        c = _draw(rng)
        w = work(c)
        # No more than the largest listed case, whatever path computes it: its
        # time is about 1 ms, which slower forms reach at fewer operations.
        aligned = all(n % 8 == 0 for _, d in _eqs(c) for n in d.values()) if c["family"] != "linattn" else True
        flops = (4e11 if aligned else 1e11) if c["dtype"] == "float16" else 5e10
        if w["bytes"] <= 1.5e9 and w["flops"] <= flops:
            return c


def _draw(rng):
    fam = rng.choice(["matmul", "matmul", "batched", "attention", "decode", "matvec", "multi_axis", "chunk", "product",
                      "linattn"])
    dtype = rng.choice(["float16", "float32"])
    if fam == "matmul":
        eq = rng.choice(["ij,jk->ik", "ij,kj->ik", "ji,jk->ik", "ji,kj->ik", "ij,jk->ki"])
        d = {c: _size(rng, 32, 8192) for c in "ijk"}
    elif fam == "batched":
        eq = rng.choice(["bji,bjk->bik", "bij,bjk->bik", "bij,bkj->bik", "bji,bkj->bik"])
        d = dict(b=_size(rng, 2, 64), **{c: _size(rng, 32, 2048) for c in "ijk"})
    elif fam == "attention":
        eq = rng.choice(["bshd,bthd->bsht", "bsht,bthd->bshd", "bhsd,bhtd->bhst", "bhst,bhtd->bhsd"])
        d = dict(b=rng.randint(1, 4), s=_size(rng, 64, 2048), t=_size(rng, 64, 2048), h=rng.choice([4, 8, 12, 16, 32]),
                 d=rng.choice([32, 64, 72, 80, 96, 128]))
    elif fam == "decode":
        return dict(family=fam, b=_size(rng, 1, 32), h=rng.choice([4, 8, 12, 16, 32]), t=_size(rng, 64, 8192),
                    d=rng.choice([32, 64, 72, 80, 96, 128]), dtype=dtype)
    elif fam == "matvec":
        eq = rng.choice(["ij,j->i", "i,ij->j", "i,ij->j", "bi,bi->b", "i,i->"])
        d = {c: _size(rng, 64, 16384) for c in "bij" if c in eq}
        if eq == "i,i->":
            d["i"] = _size(rng, 256, 1 << 22)
    elif fam == "multi_axis":
        eq = rng.choice(["ikj,jlk->il", "xyz,zyw->wx", "abc,cd->adb", "bshd,hdk->bshk", "bshd,hde->bse"])
        if eq in ("ikj,jlk->il", "xyz,zyw->wx"):
            con, free = ("kj", "il") if eq[0] == "i" else ("yz", "xw")
            d = {**{c: _size(rng, 4, 128) for c in con}, **{c: _size(rng, 32, 2048) for c in free}}
        elif eq == "abc,cd->adb":
            d = dict(a=_size(rng, 2, 128), b=_size(rng, 16, 1024), c=_size(rng, 32, 1024), d=_size(rng, 32, 1024))
        else:
            d = dict(b=rng.randint(1, 4), s=_size(rng, 16, 2048), h=rng.choice([4, 8, 12, 16]),
                     d=rng.choice([32, 64, 72, 80, 96, 128]))
            d["k" if "k" in eq else "e"] = _size(rng, 32, 2048)
    elif fam == "chunk":
        return dict(family=fam, b=_size(rng, 1, 64), h=rng.choice([2, 4, 8, 16, 32, 48]), n=rng.choice([32, 64, 128]),
                    d=rng.choice([32, 64, 128]), dtype=dtype)
    elif fam == "product":
        eq = rng.choice(["ts,ts->ts", "bsd,d->bsd", "bsd,sd->bsd", "bshd,sd->bshd", "hqk,h->hqk", "i,j->ij",
                         "st,ts->ts"])
        hi = {1: 16384, 2: 8192, 3: 2048, 4: 1024}[len(_split(eq)[2])]
        d = {c: _size(rng, 64, hi) if c not in "bh" else rng.randint(1, 32) for c in eq if c.isalpha()}
    else:
        return dict(family=fam, t=_size(rng, 64, 8192), s=_size(rng, 64, 8192), n=rng.choice([16, 32, 64, 72, 100, 128]),
                    p=_size(rng, 16, 256), dtype=dtype, precise=rng.random() < 0.25)
    return dict(family=fam, eq=eq, dims=_text(eq, d), dtype=dtype)


# ------------------------------------------------------------------- inputs --

def _decay(t, s, gamma=0.995):
    """Causal decay mask gamma^(t - s) for s <= t, else 0."""
    d = torch.arange(t, device=DEV)[:, None] - torch.arange(s, device=DEV)[None, :]
    return torch.where(d >= 0, gamma ** d.clamp(min=0).float(), torch.zeros((), device=DEV))


def _rotary(s, d):
    """cos(position * 10000^(-2i/d))."""
    pos = torch.arange(s, device=DEV, dtype=torch.float64)[:, None]
    i = torch.arange(d, device=DEV, dtype=torch.float64)[None, :] % max(1, d // 2)
    return torch.cos(pos * 10000.0 ** (-2.0 * i / d))


def _normal(g, shape, scale, dt):
    return (torch.randn(shape, generator=g, device=DEV) * scale).to(dt)


def _operands(case, seed):
    """Operand pairs of an einsum case, one for each of its equations."""
    g = torch.Generator(device=DEV).manual_seed(int(seed) * 1000003 + 17)
    dt, out = DTYPES[case["dtype"]], []
    for eq, d in _eqs(case):
        s0, s1, so = _split(eq)
        sh0, sh1 = [d[c] for c in s0], [d[c] for c in s1]
        if eq in ("bsht,bthd->bshd", "bhst,bhtd->bhsd", "bht,bthd->bhd"):
            # probabilities against values
            a = torch.softmax(torch.randn(sh0, generator=g, device=DEV), dim=-1).to(dt)
            b = _normal(g, sh1, 1.0, dt)
        elif case["family"] == "product":
            a = _normal(g, sh0, 1.0, dt)
            if eq == "bshd,sd->bshd":
                b = _rotary(d["s"], d["d"]).to(dt)
            elif eq in ("ts,ts->ts",):
                b = _decay(d["t"], d["s"]).to(dt)
            else:
                b = (torch.rand(sh1, generator=g, device=DEV) + 0.5).to(dt)
        elif eq == "i,i->":
            # values against weights, all positive: a sum well away from zero
            a, b = (torch.rand(sh, generator=g, device=DEV).to(dt) for sh in (sh0, sh1))
        elif case["family"] in ("attention", "decode", "chunk"):
            a, b = (_normal(g, sh, d["d"] ** -0.5, dt) for sh in (sh0, sh1))
        else:
            # activations against weights scaled by their fan-in
            fan = prod(d[c] for c in set(s0) & set(s1) - set(so))
            a, b = _normal(g, sh0, 1.0, dt), _normal(g, sh1, fan ** -0.5, dt)
        out.append((eq, a, b))
    return out


def _chain(case, seed):
    g = torch.Generator(device=DEV).manual_seed(int(seed) * 1000003 + 29)
    dt, t, s, n, p = DTYPES[case["dtype"]], case["t"], case["s"], case["n"], case["p"]
    q, k = _normal(g, (t, n), n ** -0.5, dt), _normal(g, (s, n), n ** -0.5, dt)
    return q, k, _normal(g, (s, p), 1.0, dt), _decay(t, s)


def prepare(case, seed):
    if case["family"] == "linattn":
        return dict(kind="chain", args=_chain(case, seed), precise=case["precise"])
    ops = _operands(case, seed)
    if case["family"] == "matmul":
        return dict(kind="einsum", args=ops[0])
    return dict(kind="runners", args=[(EinsumBuilder(eq, [tuple(a.shape), tuple(b.shape)], a.dtype).build(), a, b)
                                      for eq, a, b in ops])


def run(state):
    if state["kind"] == "chain":
        return linear_attention(*state["args"], precise=state["precise"])
    if state["kind"] == "einsum":
        return einsum(*state["args"])
    return [runner(a, b) for runner, a, b in state["args"]]


# ------------------------------------------------- work, tolerance and truth --

def work(case):
    es = 4 if case["dtype"] == "float32" else 2
    if case["family"] == "linattn":
        t, s, n, p = case["t"], case["s"], case["n"], case["p"]
        return dict(bytes=es * (t * n + s * n + s * p) + 4 * t * s + 4 * t * p, flops=2 * t * s * (n + p) + t * s)
    nbytes = flops = 0
    for eq, d in _eqs(case):
        s0, s1, so = _split(eq)
        n0, n1, no = (prod(d[c] for c in x) for x in (s0, s1, so))
        con = prod(d[c] for c in set(s0) & set(s1) - set(so))
        nbytes += es * (n0 + n1) + 4 * no
        flops += (2 if case["family"] != "product" else 1) * no * con
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    # Products are one float32 multiplication an output.  Sums are float32
    # sums of products that float32 holds exactly (float16 operands) or rounds
    # once (float32 operands).  Against 64 bits over 150 drawn cases the
    # largest relative errors were 1.4e-6 (float32; largest single one 9.4e-6)
    # and 5.7e-7 (float16; 5.7e-6); long dot products of positive values,
    # whose running sum outgrows its terms, 4e-5 at 2^24 terms, 1e-5 at 2^22.
    if case["family"] == "product":
        return "exact"
    if case["family"] == "matvec" and case["eq"] == "i,i->":
        return {"rel": 4e-5}
    return {"rel": 6e-6, "max": 4e-5} if case["dtype"] == "float32" else {"rel": 2.5e-6, "max": 2.5e-5}


def exact(case, seed):
    if case["family"] == "linattn":
        q, k, v, m = (x.double() for x in _chain(case, seed))
        return ((q @ k.t()) * m) @ v
    got = []
    for eq, a, b in _operands(case, seed):
        got.append(torch.einsum(eq, a.double(), b.double()))
    return got[0] if case["family"] == "matmul" else got
