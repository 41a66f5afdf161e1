"""The work that users of this framework have it do, as cases to be timed.

Every case goes through the Python host API on one context, as a program that
keeps its context does, and returns the histograms it gets whole.  The inputs
of a pass are the multipliers, word streams and seeds that `prepare` draws:
another seed is another code or another stream of words.

Kinds:
  an     one exhaustive AN distance distribution, A*i for i < words
  batch  the exhaustive distributions of many codes in one call
  ham    Extended Hamming weight histograms, one or several word streams a call
  mc     AN Monte Carlo, every word against m samples
  grid   the reference's grid approximation, every word (or a grid of words)
         against m samples
"""
import itertools
import random

import numpy as np

import coding_reliability_amd as cra

_CTX = None


def _context():
    """The program's context: made once, kept for all its calls."""
    global _CTX
    if _CTX is None:
        _CTX = cra.Context(0)
    return _CTX


def listed():
    return [
        # one short code, the reference's smallest recorded size: what a single call costs
        {"name": "an_a16_k8", "kind": "an", "abits": 16, "words": 1 << 8, "stride": 1},
        # the 16-bit code at 16 data bits: 32-bit codewords, 2^31 pairs
        {"name": "an_a16_k16", "kind": "an", "abits": 16, "words": 1 << 16, "stride": 1},
        # the reference's most recorded shape: a 6-bit multiplier at 24 data bits
        {"name": "an_a6_k24", "kind": "an", "abits": 6, "words": 1 << 24, "stride": 1},
        # the largest exhaustive code of the benchmark: 40-bit codewords, 2^47 pairs
        {"name": "an_a16_k24", "kind": "an", "abits": 16, "words": 1 << 24, "stride": 1},
        # the exact distribution at 32 data bits that the reference's grids approximate
        {"name": "an_a6_k32", "kind": "an", "abits": 6, "words": 1 << 32, "stride": 1},
        # the integer-stride grid of the served mix: every 4097th word of 2^32, a ragged 1048321 of them
        {"name": "an_a16_stride4097", "kind": "an", "abits": 16, "words": 1048321, "stride": 4097},
        # a quarter of the batched configuration: uneven codes of 8 to 18 data bits
        {"name": "batch_mixed", "kind": "batch", "ncodes": 1024, "kmin": 8, "kmax": 18, "abits": 16, "sweep": False},
        # the super-A sweep at 8 data bits: every odd 16-bit multiplier
        {"name": "batch_sweep_k8", "kind": "batch", "ncodes": 16384, "kmin": 8, "kmax": 8, "abits": 16, "sweep": True},
        # a share of the exhaustive (39,32) weights, as a program that splits the 2^32 words takes it
        {"name": "ham_range_k32", "kind": "ham", "k": 32, "source": "range", "count": 1 << 30, "extra": 0},
        # (39,32): the 2^34-word Monte Carlo with the 2^20-word stride grid in the same call
        {"name": "ham_mc_grid_k32", "kind": "ham", "k": 32, "source": "mc", "count": 1 << 34, "extra": 1 << 20},
        # the Monte Carlo mode at 16 data bits with the sample count of the recorded grids
        {"name": "mc_a6_n16", "kind": "mc", "abits": 6, "n": 16, "m": 10000},
        # the reference's one-dimensional grid at 32 data bits
        {"name": "grid1_a6_n32", "kind": "grid", "gdim": 1, "abits": 6, "n": 32, "m1": 1001, "m2": 0},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choice(["an", "an", "an", "batch", "ham", "ham", "mc", "grid"])
    if kind == "an":
        abits = rng.randint(3, 16)
        how = rng.choice(["full", "full", "ragged", "stride"])
        if how == "full":
            # up to 40-bit codewords, 38-bit ones beyond 24 data bits
            k = rng.randint(8, 24) if abits > 12 or rng.random() < 0.7 else rng.randint(25, min(32, 38 - abits))
            return {"kind": "an", "abits": abits, "words": 1 << k, "stride": 1}
        words = _log_int(rng, 1 << 6, 1 << 20) | 1
        return {"kind": "an", "abits": abits, "words": words, "stride": 1 if how == "ragged" else rng.randint(2, 1 << 13)}
    if kind == "batch":
        if rng.random() < 0.5:
            kmin = rng.randint(4, 12)
            return {"kind": "batch", "ncodes": _log_int(rng, 16, 4096), "kmin": kmin, "kmax": rng.randint(kmin + 1, 16),
                    "abits": rng.randint(8, 16), "sweep": False}
        abits, k = rng.randint(6, 16), rng.randint(4, 13)
        return {"kind": "batch", "ncodes": _log_int(rng, 8, 1 << (abits - 2)), "kmin": k, "kmax": k, "abits": abits,
                "sweep": True}
    if kind == "ham":
        source = rng.choice(["range", "stride", "list", "mc"])
        k = rng.randint(20, 64)
        most = {"range": min(1 << 32, 1 << k), "stride": 1 << 30, "list": 1 << 20, "mc": 1 << 32}[source]
        return {"kind": "ham", "k": k, "source": source, "count": _log_int(rng, 1 << 10, most),
                "extra": rng.choice([0, 0, _log_int(rng, 1 << 8, 1 << 20)])}
    if kind == "mc":
        n = rng.randint(8, 20)
        return {"kind": "mc", "abits": rng.randint(3, 16), "n": n, "m": _log_int(rng, 100, min(100000, 1 << (34 - n)))}
    if rng.random() < 0.5:
        n = rng.randint(16, 30)
        return {"kind": "grid", "gdim": 1, "abits": rng.randint(3, 16), "n": n,
                "m1": _log_int(rng, 101, min(100001, 1 << (40 - n), 1 << n)), "m2": 0}
    n = rng.randint(20, 32)
    return {"kind": "grid", "gdim": 2, "abits": rng.randint(3, 16), "n": n, "m1": _log_int(rng, 101, 100001),
            "m2": _log_int(rng, 101, 100001)}


def _odd(seed, bits):
    """An odd multiplier of exactly `bits` bits (3 or more): neighbouring seeds
    give different ones, also where there are only a few."""
    return (1 << (bits - 1)) | (2 * (seed * 0x9E3779B1 % (1 << (bits - 2)))) | 1


def _codes(case, rng):
    lo, bits = 1 << (case["abits"] - 1), case["abits"]
    if case["sweep"]:
        return [(A, 1 << case["kmin"]) for A in rng.sample(range(lo + 1, 1 << bits, 2), case["ncodes"])]
    return [(2 * rng.randint(1, lo - 1) + 1, 1 << rng.randint(case["kmin"], case["kmax"]))
            for _ in range(case["ncodes"])]


def prepare(case, seed):
    rng = random.Random(seed * 1000003 + 17)
    state = {"ctx": _context(), "case": case}
    kind = case["kind"]
    if kind == "an":
        state["A"], state["words"] = _odd(seed, case["abits"]) * case["stride"], case["words"]
    elif kind == "batch":
        state["codes"] = _codes(case, rng)
    elif kind == "ham":
        k, n = case["k"], case["count"]
        if case["source"] == "range":
            req = {"k": k, "source": cra.HAM_RANGE, "first": rng.randrange((1 << k) - n + 1), "count": n}
        elif case["source"] == "stride":
            req = {"k": k, "source": cra.HAM_STRIDE, "first": rng.getrandbits(16), "count": n,
                   "stride": rng.getrandbits(k - 4) | 1}
        elif case["source"] == "list":
            g = np.random.Generator(np.random.Philox(seed))
            req = {"k": k, "source": cra.HAM_LIST,
                   "words": g.integers(0, (1 << k) - 1, size=n, dtype=np.uint64, endpoint=True)}
        else:
            req = {"k": k, "source": cra.HAM_MC, "count": n, "seed": rng.getrandbits(63), "stream": 1}
        state["requests"] = [req]
        if case["extra"]:
            state["requests"].append({"k": k, "source": cra.HAM_STRIDE, "first": rng.getrandbits(16),
                                      "count": case["extra"], "stride": 65537})
    elif kind == "mc":
        state["A"], state["seed"] = _odd(seed, case["abits"]), rng.getrandbits(63)
    else:
        state["A"] = _odd(seed, case["abits"])
    return state


def run(state):
    ctx, case = state["ctx"], state["case"]
    kind = case["kind"]
    if kind == "an":
        hist, _ = ctx.an_pairs_auto(state["A"], state["words"])
    elif kind == "batch":
        rows, _ = ctx.an_batch(state["codes"])
        # the rows have as many bins as their codes need: one after the other, zeros at the end
        flat = np.fromiter(itertools.chain.from_iterable(rows), dtype=np.uint64)
        return np.pad(flat, (0, len(rows) * (case["abits"] + case["kmax"] + 1) - len(flat)))
    elif kind == "ham":
        if len(state["requests"]) > 1:
            rows, _ = ctx.hamming_weights_batch(state["requests"])
            return [np.array(row, dtype=np.uint64) for row in rows]
        hist, _ = ctx.hamming_weights(**state["requests"][0])
    elif kind == "mc":
        hist, _ = ctx.an_mc(state["A"], case["n"], case["m"], state["seed"])
    else:
        hist, _ = ctx.an_grid_ref(case["gdim"], case["n"], case["m1"], case["m2"], state["A"])
    return np.array(hist, dtype=np.uint64)


def _an_ops(abits, words):
    # words whose product has left the same carry are alike from there on: at
    # most 2^abits classes, and a histogram counts unordered pairs
    classes = min(words, 1 << abits)
    return classes * (classes + 1) // 2


def work(case):
    """Integer operations and bytes that no method can do without, one
    operation for each pair or word that is its own case."""
    kind = case["kind"]
    if kind == "an":
        abits = case["abits"] + (case["stride"] - 1).bit_length()
        return {"bytes": 8 * (abits + case["words"].bit_length() + 1), "flops": _an_ops(abits, case["words"])}
    if kind == "batch":
        ks = range(case["kmin"], case["kmax"] + 1)
        mean = sum(_an_ops(case["abits"], 1 << k) for k in ks) / len(ks)
        bins = case["abits"] + sum(ks) / len(ks) + 1
        return {"bytes": int(case["ncodes"] * (16 + 8 * bins)), "flops": int(case["ncodes"] * mean)}
    if kind == "ham":
        # consecutive words follow from the code's 2^7 dual words, block by block
        words = (64 << 7) if case["source"] == "range" else case["count"]
        read = 8 * case["count"] if case["source"] == "list" else 32
        return {"bytes": read + 8 * 72, "flops": words + case["extra"]}
    if kind == "mc":
        return {"bytes": 8 * 65, "flops": case["m"] << case["n"]}
    rows = min(1 << case["n"], case["m2"] or 1 << case["n"], 1 << (case["abits"] if case["gdim"] == 1 else 64))
    return {"bytes": 8 * 65, "flops": rows * case["m1"]}


def exact(case, seed):
    """Short codes pair by pair; the counts are whole numbers throughout."""
    if case["kind"] != "an" or case["words"] > 1 << 13:
        return None
    A = prepare(case, seed)["A"]
    w = np.arange(case["words"], dtype=np.uint64) * np.uint64(A)
    out = np.zeros(((case["words"] - 1) * A).bit_length() + 1, dtype=np.uint64)
    for i in range(len(w) - 1):
        out += np.bincount(np.bitwise_count(w[i + 1:] ^ w[i]), minlength=len(out)).astype(np.uint64)
    return out
