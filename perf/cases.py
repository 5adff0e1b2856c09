"""Contractions that a user of this library runs, for timing it.

Every case goes through the Python binding of the C ABI on torch tensors in
GPU memory, as a many-body program calls it: the descriptors are built once
(prepare_*), the calls are asynchronous on torch's current stream, tensors are
column-major unless a case says otherwise, and a and b are virtual, i and j
occupied indices where the names suggest it.

Kinds (each listed case is one size of its kind, draw() gives others):
  dense    C[abij] = A[abef] B[efij], one extent for every index: the plain
           particle-particle ladder; extent 10 is a small active space, where
           launches and latency count, 24 an ordinary small molecule
  permuted C[aibj] += alpha A[aebf] B[fjei]: the ladder in the order in which a
           program that stores its integrals as (ae|bf) has it; real and
           complex (periodic systems, relativistic spinors)
  wide     C[abcd] = A[aebf] B[ecfd] with entries over eight orders of
           magnitude, as integrals and amplitudes have, in single precision
           (default), widened to double ("fp64_mfma") or FP64-accurate
           ("ozaki"): the largest calls
  ragged   six different extents and any order of the labels in each tensor:
           the general call of a program that writes formulas as it derives them
  dpd      C[abij] = A[abef] B[efij] over the symmetry-allowed blocks of a D2h
           molecule (8 irreps), PREFIX_ROW_MAJOR storage
  batch    many independent small C[abij] = A[abef] B[efij] of uneven extents
           (pairs of a local-correlation method) in one call
  indexed  C[abij] = A[abef] B[efij] with f a sparse index: only some values
           are listed in each operand
  trace    F[mi] += A[mnef] B[inef]: the one-index intermediates (F_mi, F_ae)
           of coupled cluster, few results from long sums
  dress    C[abij] += T[ak] V[kbij]: singles dressing of a four-index tensor,
           short sums into a large result
  add      B[perm] = alpha A[abcd] + beta B[perm]: permutational symmetrisation
           of amplitudes, bound by memory
"""
import itertools
import math

import torch

import tblis_amd as T

DTYPES = {"f32": torch.float32, "f64": torch.float64, "c64": torch.complex64, "c128": torch.complex128}
DPD_EXT = (12, 9, 7, 5, 11, 8, 6, 4)


def listed():
    return [
        {"name": "dense10_f64", "kind": "dense", "n": 10, "dtype": "f64"},
        {"name": "dense24_f64", "kind": "dense", "n": 24, "dtype": "f64"},
        {"name": "permuted_f64", "kind": "permuted", "v": 64, "o": 32, "dtype": "f64"},
        {"name": "permuted_c128", "kind": "permuted", "v": 64, "o": 32, "dtype": "c128"},
        {"name": "wide96_f32", "kind": "wide", "n": 96, "config": ""},
        {"name": "ragged_f32", "kind": "ragged", "dtype": "f32", "a": 37, "b": 41, "e": 29, "f": 43, "i": 23,
         "j": 31, "A": "eafb", "B": "jefi", "C": "iabj"},
        {"name": "dpd8_f64", "kind": "dpd", "scale": 1.0, "dtype": "f64"},
        {"name": "batch1024_f32", "kind": "batch", "count": 1024, "lo": 4, "hi": 40, "shapes": 7, "dtype": "f32"},
        {"name": "indexed48_f64", "kind": "indexed", "n": 48, "nf": 32, "each": 24, "shapes": 5, "dtype": "f64"},
        {"name": "trace_f64", "kind": "trace", "m": 32, "n": 32, "e": 64, "f": 64, "dtype": "f64"},
        {"name": "dress_f64", "kind": "dress", "v": 64, "o": 32, "dtype": "f64"},
        {"name": "add96_f64", "kind": "add", "n": 96, "B": "cdab", "dtype": "f64"},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _shuffled(rng, labels):
    s = list(labels)
    rng.shuffle(s)
    return "".join(s)


def draw(rng):
    kind = rng.choice(["dense", "permuted", "wide", "ragged", "dpd", "batch", "indexed", "trace", "dress", "add"])
    real = rng.choice(["f64", "f32"])
    if kind == "dense":
        return {"kind": kind, "n": rng.randint(6, 44), "dtype": rng.choice(["f64", "f64", "f32", "c128", "c64"])}
    if kind == "permuted":
        return {"kind": kind, "v": rng.randint(16, 68), "o": rng.randint(6, 36),
                "dtype": rng.choice(["f64", "f64", "f32", "c128", "c64"])}
    if kind == "wide":
        config = rng.choice(["", "", "fp64_mfma", "ozaki"])
        return {"kind": kind, "n": rng.randint(40, 64 if config else 94), "config": config}
    if kind == "ragged":
        case = {"kind": kind, "dtype": real}
        case.update({x: rng.randint(6, 46) for x in "abefij"})
        case.update(A=_shuffled(rng, "abef"), B=_shuffled(rng, "efij"), C=_shuffled(rng, "abij"))
        return case
    if kind == "dpd":
        return {"kind": kind, "scale": round(rng.uniform(0.4, 1.6), 3), "dtype": real}
    if kind == "batch":
        lo = rng.randint(2, 12)
        return {"kind": kind, "count": _log(rng, 32, 1024), "lo": lo, "hi": rng.randint(lo + 4, 40),
                "shapes": rng.randint(1, 10 ** 6), "dtype": real}
    if kind == "indexed":
        nf = rng.randint(6, 40)
        return {"kind": kind, "n": rng.randint(12, 50), "nf": nf, "each": rng.randint(nf // 2 + 1, nf),
                "shapes": rng.randint(1, 10 ** 6), "dtype": real}
    if kind == "trace":
        return {"kind": kind, "m": rng.randint(6, 64), "n": rng.randint(6, 48), "e": rng.randint(16, 72),
                "f": rng.randint(16, 72), "dtype": real}
    if kind == "dress":
        return {"kind": kind, "v": rng.randint(12, 80), "o": rng.randint(4, 40), "dtype": real}
    return {"kind": kind, "n": rng.randint(12, 94), "B": rng.choice(["badc", "cdab", "dcba", "bacd", "abdc", "acbd"]),
            "dtype": real}


# ---------------------------------------------------------------- inputs

def _colmajor(lens):
    s, a = [], 1
    for x in lens:
        s.append(a)
        a *= x
    return s


def _rand(g, n, dtype):
    """n values uniform in [-1, 1) (both parts of a complex number)."""
    real = {torch.complex64: torch.float32, torch.complex128: torch.float64}.get(dtype, dtype)
    k = 2 * n if real != dtype else n
    x = torch.rand(k, dtype=real, device="cuda", generator=g) * 2 - 1
    return torch.view_as_complex(x.reshape(n, 2)) if real != dtype else x


def _outliers(g, n, dtype):
    """normal(0, 1) with 1% of the entries scaled by 1e4."""
    x = torch.randn(n, dtype=torch.float32, device="cuda", generator=g)
    x[torch.rand(n, device="cuda", generator=g) < 0.01] *= 1e4
    return x.to(dtype)


def _view(flat, lens, at=0):
    return torch.as_strided(flat, lens, _colmajor(lens), at)


def _formula(case):
    """Labels of A, B, C, the extent of each label, alpha, beta."""
    kind = case["kind"]
    if kind == "dense":
        return "abef", "efij", "abij", dict.fromkeys("abefij", case["n"]), 1.0, 0.0
    if kind == "permuted":
        v, o = case["v"], case["o"]
        alpha = 0.5 + 0.25j if case["dtype"][0] == "c" else 0.5
        return "aebf", "fjei", "aibj", dict(a=v, b=v, e=v, f=v, i=o, j=o), alpha, 1.0
    if kind == "wide":
        return "aebf", "ecfd", "abcd", dict.fromkeys("abcdef", case["n"]), 1.0, 0.0
    if kind == "ragged":
        return case["A"], case["B"], case["C"], {x: case[x] for x in "abefij"}, -1.0, 0.0
    if kind == "trace":
        return "mnef", "inef", "mi", dict(m=case["m"], i=case["m"], n=case["n"], e=case["e"], f=case["f"]), 0.5, 1.0
    assert kind == "dress"
    v, o = case["v"], case["o"]
    return "ak", "kbij", "abij", dict(a=v, b=v, i=o, j=o, k=o), -1.0, 1.0


def _dtype(case):
    if case["kind"] == "wide":  # the FP64-accurate mode is for values held in double
        return torch.float64 if case["config"] == "ozaki" else torch.float32
    return DTYPES[case["dtype"]]


def _dpd_lens(case):
    return [max(1, int(round(x * case["scale"]))) for x in DPD_EXT]


def _batch_shapes(case):
    import random
    rng = random.Random(case["shapes"])
    shapes, at = [], [0, 0, 0]
    for _ in range(case["count"]):
        a, b, e, f, i, j = (rng.randint(case["lo"], case["hi"]) for _ in range(6))
        row = [(lens, at[t]) for t, lens in enumerate(([a, b, e, f], [e, f, i, j], [a, b, i, j]))]
        for t in range(3):
            at[t] += math.prod(row[t][0])
        shapes.append(row)
    return shapes, at


def _listed_values(case):
    import random
    rng = random.Random(case["shapes"])
    return [sorted(rng.sample(range(case["nf"]), case["each"])) for _ in range(2)]


def _inputs(case, seed):
    """The flat buffers of A, B and C (C: what it holds before the call)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind, dtype = case["kind"], _dtype(case)
    if kind == "dpd":
        n = _dpd_size(_dpd_lens(case))
        return [_rand(g, n, dtype), _rand(g, n, dtype), torch.zeros(n, dtype=dtype, device="cuda")]
    if kind == "batch":
        at = _batch_shapes(case)[1]
        return [_rand(g, at[0], dtype), _rand(g, at[1], dtype), torch.zeros(at[2], dtype=dtype, device="cuda")]
    if kind == "indexed":
        n3 = case["n"] ** 3 * case["each"]
        return [_rand(g, n3, dtype), _rand(g, n3, dtype), torch.zeros(case["n"] ** 4, dtype=dtype, device="cuda")]
    if kind == "add":
        return [_rand(g, case["n"] ** 4, dtype), _rand(g, case["n"] ** 4, dtype)]
    la, lb, lc, ext, _, beta = _formula(case)
    na, nb, nc = (math.prod(ext[x] for x in s) for s in (la, lb, lc))
    make = _outliers if kind == "wide" else _rand
    return [make(g, na, dtype), make(g, nb, dtype),
            _rand(g, nc, dtype) if beta else torch.zeros(nc, dtype=dtype, device="cuda")]


def prepare(case, seed):
    T.set_stream(torch.cuda.current_stream().cuda_stream)
    T.set_async(True)
    kind = case["kind"]
    bufs = _inputs(case, seed)
    A, B = bufs[0], bufs[1]
    if kind == "add":
        lens = [case["n"]] * 4
        a, b = _view(A, lens), _view(B, lens)
        return {"call": lambda: T.add(0.5, a, "abcd", 0.5, b, case["B"]), "out": B}
    C = bufs[2]
    if kind == "dpd":
        lens = [_dpd_lens(case)] * 4
        call = T.prepare_dpd_mult(1.0, A, 0, "abef", B, 0, "efij", 0.0, C, 0, "abij", 8, lens, lens, lens)
    elif kind == "batch":
        shapes = _batch_shapes(case)[0]
        ops = [[_view(bufs[t], row[t][0], row[t][1]) for row in shapes] for t in range(3)]
        n = len(shapes)
        call = T.prepare_batch(1.0, ops[0], ["abef"] * n, ops[1], ["efij"] * n, 0.0, ops[2], ["abij"] * n)
    elif kind == "indexed":
        n = case["n"]
        fa, fb = _listed_values(case)
        xa, xb = ([_view(x, [n] * 3, k * n ** 3) for k in range(case["each"])] for x in (A, B))
        call = T.prepare_indexed_mult(1.0, T.Indexed(xa, [(f,) for f in fa], [case["nf"]]), "abef",
                                      T.Indexed(xb, [(f,) for f in fb], [case["nf"]]), "eijf", 0.0,
                                      T.Indexed([_view(C, [n] * 4)], [()], []), "abij")
    else:
        la, lb, lc, ext, alpha, beta = _formula(case)
        va, vb, vc = (_view(x, [ext[c] for c in s]) for x, s in ((A, la), (B, lb), (C, lc)))
        call = T.prepare_mult(alpha, va, la, vb, lb, beta, vc, lc, config=case.get("config") or None)
    return {"call": call, "out": C}


def run(state):
    state["call"]()
    return state["out"]


# ---------------------------------------------------------------- work

def _dpd_prefix(lens):
    """Elements of the first k dimensions together, by their irrep product."""
    size = [list(lens)]
    for _ in range(3):
        size.append([sum(size[-1][r ^ s] * lens[s] for s in range(8)) for r in range(8)])
    return size


def _dpd_size(lens):
    return _dpd_prefix(lens)[3][0]


def work(case):
    kind, dtype = case["kind"], _dtype(case)
    e = torch.empty(0, dtype=dtype).element_size()
    mul = 8.0 if dtype.is_complex else 2.0
    if kind == "dpd":
        lens = _dpd_lens(case)
        s = [sum(lens[h] * lens[h ^ r] for h in range(8)) for r in range(8)]
        return {"bytes": 3.0 * e * _dpd_size(lens), "flops": sum(2.0 * x ** 3 for x in s)}
    if kind == "batch":
        shapes, at = _batch_shapes(case)
        return {"bytes": float(e * sum(at)),
                "flops": sum(2.0 * math.prod(r[0][0]) * math.prod(r[2][0][2:]) for r in shapes)}
    if kind == "indexed":
        n, (fa, fb) = case["n"], _listed_values(case)
        match = len(set(fa) & set(fb))
        return {"bytes": float(e * (2 * match * n ** 3 + n ** 4)), "flops": 2.0 * match * n ** 5}
    if kind == "add":
        return {"bytes": 3.0 * e * case["n"] ** 4, "flops": 3.0 * case["n"] ** 4}
    la, lb, lc, ext, _, beta = _formula(case)
    na, nb, nc = (math.prod(ext[x] for x in s) for s in (la, lb, lc))
    return {"bytes": float(e * (na + nb + (2 if beta else 1) * nc)),
            "flops": mul * math.prod(ext[x] for x in set(la + lb + lc))}


# ---------------------------------------------------------------- in 64 bits

def _contract(la, a, lb, b, lc):
    """Two operands' contraction as one matrix product."""
    k = [x for x in la if x in lb]
    m, n = [x for x in la if x not in k], [x for x in lb if x not in k]
    am = a.permute([la.index(x) for x in m + k])
    bm = b.permute([lb.index(x) for x in k + n])
    sizes = list(am.shape[:len(m)]) + list(bm.shape[len(k):])
    kk = math.prod(bm.shape[:len(k)])
    c = am.reshape(-1, kk) @ bm.reshape(kk, -1)
    return c.reshape(sizes).permute([(m + n).index(x) for x in lc])


def _flat(x):
    """The column-major storage of a tensor."""
    return x.permute(*range(x.dim() - 1, -1, -1)).reshape(-1)


def _dpd_blocks(flat, lens):
    """PREFIX_ROW_MAJOR: dimensions in reversed order, the first fastest; the
    blocks of each prefix follow one another by the irrep of its last dimension."""
    size = _dpd_prefix(lens)
    out = {}
    for r in itertools.product(range(8), repeat=4):
        if r[0] ^ r[1] ^ r[2] ^ r[3]:
            continue
        q = r[::-1]
        at, total, stride = 0, 0, [1, 0, 0, 0]
        for d in (3, 2, 1):
            at += sum(size[d - 1][s ^ total] * lens[s] for s in range(q[d]))
            total ^= q[d]
            stride[d] = size[d - 1][total]
        out[r] = torch.as_strided(flat, [lens[x] for x in r], stride[::-1], at)
    return out


def exact(case, seed):
    kind = case["kind"]
    wide = torch.complex128 if _dtype(case).is_complex else torch.float64
    bufs = [x.to(wide) for x in _inputs(case, seed)]
    A, B = bufs[0], bufs[1]
    if kind == "add":
        lens = [case["n"]] * 4
        a, b = _view(A, lens), _view(B, lens)
        return _flat(0.5 * a.permute(["abcd".index(x) for x in case["B"]]) + 0.5 * b)
    C = bufs[2]
    if kind == "dpd":
        lens = _dpd_lens(case)
        a, b, c = (_dpd_blocks(x, lens) for x in (A, B, C))
        for r, out in c.items():
            for e in range(8):
                f = r[0] ^ r[1] ^ e
                out += _contract("abef", a[r[0], r[1], e, f], "efij", b[e, f, r[2], r[3]], "abij")
        return C
    if kind == "batch":
        for row in _batch_shapes(case)[0]:
            a, b, c = (_view(bufs[t], row[t][0], row[t][1]) for t in range(3))
            c.copy_(_contract("abef", a, "efij", b, "abij"))
        return C
    if kind == "indexed":
        n, (fa, fb) = case["n"], _listed_values(case)
        out = torch.zeros([n] * 4, dtype=wide, device="cuda")
        for f in sorted(set(fa) & set(fb)):
            out += _contract("abe", _view(A, [n] * 3, fa.index(f) * n ** 3), "eij",
                             _view(B, [n] * 3, fb.index(f) * n ** 3), "abij")
        return _flat(out)
    la, lb, lc, ext, alpha, beta = _formula(case)
    a, b, c = (_view(x, [ext[y] for y in s]) for x, s in ((A, la), (B, lb), (C, lc)))
    out = alpha * _contract(la, a, lb, b, lc)
    return _flat(out + beta * c if beta else out)
