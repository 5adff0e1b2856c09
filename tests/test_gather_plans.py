"""The tables of the gather tiles (tblis_hip_debug_plan) on the host: every
address that the kernels form from them, in their own 32- and 64-bit
arithmetic, lies inside its operand and on the boundary its load needs, and
the products at these addresses are the contraction.  Inputs are small whole
numbers, so the comparison is exact."""
import ctypes as C
import itertools
import os
import subprocess
import sys
import time

import numpy as np
import pytest

import tblis_amd as T
from tests.test_boundary import _HostDesc

HEADER = 24  # TBLIS_HIP_PLAN_HEADER
F64, F32, C64, C128 = T.TYPE_DOUBLE, T.TYPE_SINGLE, T.TYPE_SCOMPLEX, T.TYPE_DCOMPLEX


class Plan:
    """A plan of C = A B over tensors given as (lengths, strides, labels)."""

    CAP = 1 << 22

    def __init__(self, A, B, C_, dtype=F64, aligned=True, config=None, data=16):
        d = [_HostDesc(x[0], x[1], dtype) for x in (A, B, C_)]
        for t in d:
            t.d.data = C.c_void_p(data)  # (never read)
        args = [y for t, x in zip(d, (A, B, C_)) for y in (C.byref(t.d), x[2].encode("latin1"))]
        cap = self.CAP
        out = np.zeros(cap, dtype=np.int64)
        n = T.lib().tblis_hip_debug_plan(T.get_config(config) if config else None, *args, int(aligned),
                                         out.ctypes.data_as(C.POINTER(C.c_int64)), cap)
        assert n >= HEADER, (n, T.last_error())
        (self.tile, self.gather, self.pieces, self.slices, self.swap, self.bk, self.bm, self.bn, self.elem,
         self.family, nt, nu, npool, self.scaled) = (int(x) for x in out[:14])
        self.key = int(out[23]) & ((1 << 64) - 1)
        self.groups = {g: int(x) for g, x in enumerate(out[14:23]) if x}
        if self.gather:
            at = HEADER
            self.tasks = out[at:at + 16 * nt].reshape(nt, 16)
            at += 16 * nt
            self.sums = out[at:at + 8 * nu].reshape(nu, 8)
            self.pool = out[at + 8 * nu:n].copy()
            assert len(self.pool) == npool

    def loads(self, o, t, data, lo):
        """Operand o's tile of task t as the kernel reads it from data, whose
        first element is element lo of the tensor."""
        group, kbeg, kend = (int(x) for x in t[:3])
        src, rt, km = (int(t[3 + o + 2 * i]) for i in range(3))
        valid = int(t[10 + o])
        f64 = self.family == 0
        mode = (group >> o) & 1 if f64 else group // 3 ** o % 3
        size = self.bm if o == 0 else self.bn
        nk = kend - kbeg
        stages = -(-nk // self.bk)
        # the kernels load up to a stage past the end
        k = np.arange((stages + (0 if self.pieces else 1)) * self.bk)
        r = np.arange(size)
        wrap = (1 << 32) - 1
        ks = self.pool[km:] if f64 else self.pool[km:].view(np.uint32).astype(np.int64)
        ks = ks[kbeg:]
        row = lambda r: self.pool[rt + np.where(r < valid, r, 0)]
        if self.pieces:
            first = ks[k - k % self.bk]
            lead = k % self.bk if not mode else k % self.bk - k % self.bk % 2
            delta = (ks[np.where(lead < nk, lead, 0)] - ks[0]) & wrap
            rows = row(r - r % 2 if not mode else r)
            at = first + (((rows & wrap)[:, None] + delta) & wrap)
            keep = k < nk
            assert (at[:, keep] + src * 8 >= lo * 8).all() and ((at[:, keep] + src * 8) % 16 == 0).all()
            at += 8 * ((r % 2)[:, None] if not mode else k % 2)
            at, k = at[:, keep], k[keep]
        else:
            assert (ks[:len(k)] >= 0).all() and (ks[:len(k)] <= wrap).all()
            at = row(r)[:, None] + (ks[k] if mode < 2 else ks[k - k % 8])
            assert (at >= 0).all() and (at <= wrap).all()
            if mode == 2:
                assert ((at + src * 4) % 16 == 0).all()
                at = at + 4 * (k % 8)
        at = at + src * self.elem
        assert (at % self.elem == 0).all()
        at = at // self.elem - lo
        assert (at >= 0).all() and (at < len(data)).all(), (at.min(), at.max(), len(data))
        return data[at][:valid, :nk]

    def run(self, a, b, c):
        """C += A B on host arrays (each: data, lo) through the plan's tables."""
        ops = (b, a) if self.swap else (a, b)
        slices = np.zeros(sum(int(u[4] * u[5] * u[6]) for u in self.sums))
        for t in self.tasks:
            x, y = (self.loads(o, t, *ops[o]) for o in range(2))
            if self.scaled:
                x = x * self.pool[int(t[9]) + int(t[1]):][:x.shape[1]].view(np.float64)
            p = x @ y.T
            i, j = (np.arange(int(t[10 + o])) for o in range(2))
            if t[15]:
                slices[int(t[12]) + i[:, None] * int(t[15]) + j] = p
            else:
                self.store(c, t[12:15], p)
        for u in self.sums:
            m, n = int(u[4]), int(u[5])
            p = sum(slices[int(u[3]) + s * int(u[7]):][:m * n] for s in range(int(u[6])))
            self.store(c, u[:3], p.reshape(m, n))

    def store(self, c, at, p):
        data, lo = c
        i, j = (np.arange(x) for x in p.shape)
        at = int(at[0]) + self.pool[int(at[1]) + i][:, None] + self.pool[int(at[2]) + j] - lo
        assert (at >= 0).all() and (at < len(data)).all()
        data[at] += p


def _span(lens, strides):
    reach = [(n - 1) * s for n, s in zip(lens, strides)]
    return sum(min(x, 0) for x in reach), sum(max(x, 0) for x in reach)


def _check(A, B, C_, dtype=F64, **kw):
    """The plan's products against numpy's; returns the plan."""
    plan = Plan(A, B, C_, dtype, **kw)
    if not plan.gather:
        return plan
    parts = 2 if dtype in (C64, C128) else 1
    rng = np.random.default_rng(1)
    flat, view = [], []
    for lens, strides, _ in (A, B, C_):
        lo, hi = _span(lens, strides)
        x = rng.integers(-4, 5, size=parts * (hi - lo + 1)).astype(np.float64)
        flat.append((x, parts * lo))
        x = x.view(np.complex128) if parts == 2 else x
        view.append(np.lib.stride_tricks.as_strided(x[-lo:], lens, [s * x.itemsize for s in strides]))
    want = np.array(view[2]) + np.einsum(f"{A[2]},{B[2]}->{C_[2]}", view[0], view[1])
    plan.run(*flat)
    assert (np.array(view[2]) == want).all()
    return plan


def _packed(lens):
    return [int(np.prod(lens[:i])) for i in range(len(lens))]


def _tensor(ext, labels, negative="", gap=1):
    """Packed in the order of the labels (gap: of the first stride), the
    strides of `negative` turned round."""
    lens = [ext[x] for x in labels]
    return lens, [(-s if x in negative else s) * gap for s, x in zip(_packed(lens), labels)], labels


@pytest.mark.parametrize("dtype", [F64, F32])
@pytest.mark.parametrize("negA,negB", [("k", ""), ("", "k"), ("k", "k"), ("a", ""), ("ak", "b"), ("ak", "bk")])
@pytest.mark.parametrize("A,B", [("ak", "kb"), ("ka", "kb"), ("ak", "bk"), ("ka", "bk")])
def test_negative_strides(A, B, negA, negB, dtype):
    """Rows, k or both of an operand in descending order, on extents that
    allow 16-byte pieces when they ascend."""
    for ext in (dict(a=64, b=64, k=64), dict(a=34, b=66, k=80), dict(a=8, b=8, k=4096)):
        plan = _check(_tensor(ext, A, negA), _tensor(ext, B, negB), _tensor(ext, "ab"), dtype)
        if dtype == F64 and not negA + negB:
            assert plan.pieces


@pytest.mark.parametrize("dtype", [F64, F32])
def test_negative_strides_in_two_dimensions_of_k(dtype):
    """k = (e, f): either of them descending, in both operands or in one."""
    ext = dict(a=32, e=16, f=6, b=34)
    for negA, negB in itertools.product(["", "e", "f", "ef"], repeat=2):
        for A, B in (("aef", "efb"), ("efa", "bfe"), ("eaf", "ebf")):
            plan = _check(_tensor(ext, A, negA), _tensor(ext, B, negB), _tensor(ext, "ab"), dtype)
            assert plan.gather or (negA + negB)


@pytest.mark.parametrize("seed", range(60))
def test_forms_of_the_general_path(seed, monkeypatch):
    """Orders of the labels, gaps, negative and zero strides, odd extents,
    every gather tile and number of slices, aligned tensors or not."""
    rng = np.random.default_rng(8000 + seed)
    ran = 0
    for dtype, tiles in ((F64, "9 10 11"), (F32, "6 7"), (C128, "9 10 11")):
        for tile in tiles.split():
            monkeypatch.setenv("TBLIS_HIP_PANEL_TILE", tile)
            monkeypatch.setenv("TBLIS_HIP_KSPLIT", str(rng.choice([1, 1, 2, 3])))
            ext = {x: int(rng.choice([1, 2, 3, 4, 5, 8, 16, 17])) for x in "abij"}
            ext.update({x: int(rng.choice([1, 2, 3, 7, 8, 16, 32])) for x in "ef"})
            form = []
            for labels in ("abef", "efij", "abij"):
                s = "".join(rng.permutation(list(labels)))
                neg = "".join(x for x in s if rng.random() < 0.15)
                lens, strides, s = _tensor(ext, s, neg, int(rng.choice([1, 1, 1, 2])))
                if labels != "abij" and rng.random() < 0.15:
                    strides[int(rng.integers(4))] = 0
                form.append((lens, strides, s))
            plan = _check(*form, dtype, aligned=bool(rng.integers(2)))
            ran += plan.gather and plan.tile == int(tile)
    assert ran == 8


def _plans_with(path, lines, program):
    """What `program` prints, in a process whose tuning file has these
    (key, family, tile) lines."""
    path.write_text("".join('{"format": "tblis-tune-v3", "family": %d, "shapes": "%016x", "tile": %d, "packed": 0}\n'
                            % (family, key, tile) for key, family, tile in lines))
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = subprocess.run([sys.executable, "-c", "import sys; sys.path.insert(0, %r)\n" % root + program],
                         capture_output=True, text=True,
                         env=dict(os.environ, TBLIS_HIP_AUTOTUNE="1", TBLIS_HIP_TUNE_FILE=str(path)))
    assert out.returncode == 0, out.stderr
    return [[int(x) for x in line.split()] for line in out.stdout.splitlines()]


# Calls of one m, n, k whose operands have several k blocks (complex parts):
# packed tensors, and views that reach past 4 GiB, which no gather tile can
# address.
_TUNED = """
from tests.test_gather_plans import C128, Plan
small = [([32, 32], [1, 32], s) for s in ("ak", "kb", "ab")]
far = [([32, 32], [1, 1 << 25], "ak"), *small[1:]]
turned = [([32, 32], [32, 1], "ak"), *small[1:]]
for x in (small, far, turned):
    p = Plan(*x, dtype=C128)
    print(p.tile, p.gather, p.key)
"""


def test_remembered_tile_only_where_it_applies(tmp_path):
    """A gather tile from the tuning file is used where it can run, and not
    for operands beyond its reach; operands of several blocks that differ in
    their strides have lines of their own."""

    path = tmp_path / "tune.txt"
    keys = [key for _, _, key in _plans_with(path, [], _TUNED)]
    assert len(set(keys)) == 3
    small, far, turned = _plans_with(path, [(k, 0, tile) for k, tile in zip(keys, (9, 9, 3))], _TUNED)
    assert small[:2] == [9, 1] and turned[:2] == [3, 0]
    assert not far[1]


_WITHOUT_TENSORS = """
from tests.test_gather_plans import F32, Plan
p = Plan(*[([200, 200], [1, 200], s) for s in ("ak", "kb", "ab")], dtype=F32, data={data})
print(p.tile, p.gather, p.key)
"""


@pytest.mark.parametrize("data", [16, None])
def test_remembered_panel_tile_against_a_gather_tile(data, tmp_path):
    """Plans made without the tensors (indexed contractions) time panel tiles
    only, whose best one does not replace the model's gather tile; with the
    tensors it was timed against it and does."""
    path = tmp_path / "tune.txt"
    program = _WITHOUT_TENSORS.format(data=data)
    [[tile, gather, key]] = _plans_with(path, [], program)
    assert gather
    assert _plans_with(path, [(key, 1, 3)], program) == [[3, 0, key] if data else [tile, gather, key]]


@pytest.mark.parametrize("dtype", [F64, F32])
def test_planning_time_of_long_sums(dtype, monkeypatch):
    """Planning a gather tile makes each operand's tables once: 32 x 32 x
    131072 takes as long as some passes over tables of its length (FP64 15 of
    them; 60 when its models and its plan each made the tables anew)."""
    ext = dict(a=32, b=32, k=131072)
    form = [_tensor(ext, s) for s in ("ak", "kb", "ab")]
    words = np.arange(2 * ext["k"])

    def best(f):
        t = []
        for _ in range(9):
            t0 = time.perf_counter()
            f()
            t.append(time.perf_counter() - t0)
        return min(t)

    d = [_HostDesc(x[0], x[1], dtype) for x in form]
    args = [y for t, x in zip(d, form) for y in (C.byref(t.d), x[2].encode("latin1"))]
    out = (C.c_int64 * HEADER)()  # too small: the plan is made, not copied out
    plan = best(lambda: T.lib().tblis_hip_debug_plan(None, *args, 1, out, HEADER))
    one = best(lambda: (words[1:] - words[:-1]).sum() + words.copy()[0])
    assert plan <= 40 * one, (plan, one)


# (labels, extents, type, gather tile or not): both sides of the rules between
# packing and gathering, and between the orders that a gather tile walks.
# Times on an MI355X (us): 6480 x 1824 x 3328 with pairs along k packed 567,
# gathered 1164; 1972 x 1920 x 4560 in pairs 266, 530; 40320 x 2976 x 256 packed
# 1050, gathered in the other order 1695.
RULES = [
    ("gbface,gjief->iacjb", dict(a=9, b=24, c=30, i=38, j=48, e=26, f=64, g=2), F32, False),
    ("cfgbae,ikgefj->ijakbc", dict(a=34, b=29, c=2, i=2, j=32, k=30, e=5, f=57, g=16), F32, False),
    ("aebf,ecfd->abcd", dict.fromkeys("abcdef", 60), F32, False),
    ("bcefa,efji->cbija", dict(a=40, b=63, c=16, i=62, j=48, e=8, f=32), F64, False),
    ("aebf,fjei->aibj", dict(a=64, b=64, e=64, f=64, i=32, j=32), F64, True),
    ("abef,efij->abij", dict.fromkeys("abefij", 24), F64, True),
    ("abef,efij->abij", dict.fromkeys("abefij", 24), F32, True),
    ("eafb,jefi->iabj", dict(a=37, b=41, e=29, f=43, i=23, j=31), F32, True),
    ("mnef,inef->mi", dict(m=32, i=32, n=32, e=64, f=64), F64, True),
    ("ak,kbij->abij", dict(a=64, b=64, i=32, j=32, k=32), F64, True),
]


@pytest.mark.parametrize("labels,ext,dtype,gather", RULES)
def test_gathered_or_packed(labels, ext, dtype, gather):
    A, rest = labels.split(",")
    B, C_ = rest.split("->")
    assert bool(Plan(*[_tensor(ext, s) for s in (A, B, C_)], dtype=dtype).gather) == gather


def _matrix(m, n, row_major, labels):
    return [m, n], [n, 1] if row_major else [1, m], labels


SHAPES = [(32, 64, 16), (34, 66, 18), (130, 2, 130), (66, 34, 31), (33, 64, 98), (64, 130, 162), (129, 127, 47),
          (200, 8, 80), (8, 264, 1100)]


@pytest.mark.parametrize("aligned", [True, False])
@pytest.mark.parametrize("ra", [False, True])
@pytest.mark.parametrize("rb", [False, True])
def test_load_modes(ra, rb, aligned, monkeypatch):
    """FP64 pieces run where both operands' contiguous extent and the other
    stride are even and the tensors start on 16 bytes; split-BF16 loads
    aligned eights of k in mode 2, other contiguous k in mode 1, rows in
    mode 0."""
    for m, n, k in SHAPES:
        A, B, C_ = _matrix(m, k, ra, "ak"), _matrix(k, n, rb, "kb"), _matrix(m, n, True, "ab")
        even = (k if ra else m) % 2 == 0 and (n if rb else k) % 2 == 0
        for tile in ("9", "10", "11"):
            monkeypatch.setenv("TBLIS_HIP_PANEL_TILE", tile)
            p = Plan(A, B, C_, F64, aligned=aligned)
            assert (p.tile, p.pieces) == (int(tile), aligned and even), (m, n, k)
            assert list(p.groups) == [ra + 2 * (not rb)]
        eights = 2 if aligned and k % 8 == 0 else 1
        for tile in ("6", "7"):
            monkeypatch.setenv("TBLIS_HIP_PANEL_TILE", tile)
            p = Plan(A, B, C_, F32, aligned=aligned)
            assert p.tile == int(tile)
            assert list(p.groups) == [(eights if ra else 0) + 3 * (0 if rb else eights)], (m, n, k)


@pytest.mark.parametrize("dtype,elem", [(F64, 8), (F32, 4)])
@pytest.mark.parametrize("back", [1, -1])
def test_reach_of_four_gib(back, dtype, elem):
    """Offsets are 32-bit bytes: an operand that spans 4 GiB is packed, one
    that ends just below is gathered, in either direction of its stride."""
    for gather, span in ((True, (1 << 32) // elem - 2), (False, (1 << 32) // elem)):
        A = [64, 8], [1, back * ((span - 64) // 7)], "ak"
        A[1][1] += back * (0 if gather else 1)
        reach = (63 + 7 * abs(A[1][1]) + 1) * elem
        assert (reach < 1 << 32) == gather
        plan = Plan(A, _matrix(8, 64, False, "kb"), _matrix(64, 64, False, "ab"), dtype)
        assert bool(plan.gather) == gather


@pytest.mark.parametrize("m,n,k,dtype,tile", [
    (1225, 1225, 120, F64, 10), (33, 4489, 225, F64, 11), (2500, 31, 2499, F64, 11), (4489, 1225, 4489, F64, 8),
    (2025, 2025, 2025, F64, 5), (1296, 1296, 1296, F32, 7), (2561, 2049, 1700, F32, 6), (4096, 4096, 2048, F32, 0),
    (8192, 8192, 8192, F32, 0)])
def test_tiles_picked(m, n, k, dtype, tile):
    """One size of each side of the lines between tiles."""
    plan = Plan(_matrix(m, k, False, "ak"), _matrix(k, n, False, "kb"), _matrix(m, n, dtype == F32, "ab"), dtype)
    assert plan.tile == tile
