"""The gather tiles (both operands read from the tensors through LDS) and the
k slices of GEMMs with few C tiles, against the oracle.

Sizes sit where the kernels can go wrong: one row or column, tile edges and
one past them, k below, at and past a stage and a slice, slices that a short
k leaves without work, rows and k in odd strides, several k blocks with
scales (complex and indexed contractions).  FP64 bar: 1e-12 relative
Frobenius error, the repository's bound for every FP64 path (the sums here
have at most 1100 terms, whose rounding stays under 1e-13 of the norm)."""
import numpy as np
import pytest
import torch

import tblis_amd as T
from tests.test_gpu_parity import DEV, FP64_TOL, _dense_case, rel_fro

pytestmark = pytest.mark.gpu


@pytest.fixture
def plans(monkeypatch):
    """Set knobs for plans built in the test; no plan outlives it."""
    T.lib().tblis_hip_clear_plan_cache()
    yield monkeypatch
    T.lib().tblis_hip_clear_plan_cache()


@pytest.mark.parametrize("slices", ["1", "2", "5", "40"])
@pytest.mark.parametrize("tile", ["9", "10", "11"])
def test_gather_tiles_in_slices(tile, slices, plans):
    plans.setenv("TBLIS_HIP_PANEL_TILE", tile)
    plans.setenv("TBLIS_HIP_KSPLIT", slices)
    rng = np.random.default_rng(71000 + int(tile) * 100 + int(slices))
    for m, n, k in [(1, 1, 1), (1, 65, 17), (64, 1, 33), (32, 32, 16), (33, 31, 15), (65, 64, 32), (129, 127, 47),
                    (40, 24, 1100)]:
        kinds = ["col", "row", "random"]
        rng.shuffle(kinds)
        _dense_case(rng, "ak", "kb", "ab", dict(a=m, b=n, k=k), kinds, alpha=1.5, beta=-0.5)
        assert T.last_tile() == int(tile)
    # k of several dimensions in another order than the rows', odd extents
    _dense_case(rng, "eafb", "jefi", "iabj", dict(a=7, b=9, e=5, f=13, i=3, j=11), ["col"] * 3, beta=0.0)
    _dense_case(rng, "aebf", "fjei", "aibj", dict(a=12, b=10, e=9, f=11, i=7, j=13), ["col"] * 3,
                dtype=np.float32, config="fp64_mfma", tol=2e-7)


@pytest.mark.parametrize("at", [0, 1])
@pytest.mark.parametrize("slices", ["1", "3"])
@pytest.mark.parametrize("tile", ["9", "10", "11"])
def test_gather_in_pieces(tile, slices, at, plans):
    """Operands whose rows or k come in pairs are read 16 bytes at a time when
    the tensors start on 16 bytes (at 0), element by element when they do not
    (at 1): lanes along rows and along k on either side, last stages of 2 to
    BK - 2 k and of an odd number of them, an odd number of rows, k of two
    dimensions, beta = 0 over NaN."""
    plans.setenv("TBLIS_HIP_PANEL_TILE", tile)
    plans.setenv("TBLIS_HIP_KSPLIT", slices)
    g = torch.Generator(device=DEV).manual_seed(75000 + int(tile) * 10 + int(slices) + at)

    def tensor(shape, row_major):
        flat = torch.rand(at + shape[0] * shape[1], dtype=torch.float64, device=DEV, generator=g) - 0.5
        v = flat[at:]
        return v.view(shape) if row_major else v.view(shape[1], shape[0]).t()

    for m, n, k in [(2, 2, 2), (32, 64, 16), (34, 66, 18), (130, 2, 130), (66, 34, 31), (33, 64, 98), (64, 130, 162)]:
        for ra in (False, True):
            for rb in (False, True):
                A, B = tensor((m, k), ra), tensor((k, n), rb)
                C = torch.full((m, n), float("nan"), dtype=torch.float64, device=DEV)
                T.mult(1.5, A, "ak", B, "kb", 0.0, C, "ab")
                torch.cuda.synchronize()
                assert T.last_tile() == int(tile)
                want = 1.5 * (A.cpu().numpy() @ B.cpu().numpy())
                assert rel_fro(C.cpu().numpy(), want) <= FP64_TOL, (m, n, k, ra, rb)
    # k = (e, f) in stages of one dimension: 32 and 64 fill the stages
    x = torch.rand(at + 6 * 32 * 10 * 4, dtype=torch.float64, device=DEV, generator=g)[at:].view(4, 10, 32, 6) - 0.5
    y = torch.rand(at + 32 * 8 * 4 * 5, dtype=torch.float64, device=DEV, generator=g)[at:].view(5, 4, 8, 32) - 0.5
    C = torch.zeros(5, 8, 10, 6, dtype=torch.float64, device=DEV)
    T.mult(1.0, x, "fbea", y, "jfie", 0.0, C, "jiba")
    torch.cuda.synchronize()
    want = np.einsum("fbea,jfie->jiba", x.cpu().numpy(), y.cpu().numpy())
    assert rel_fro(C.cpu().numpy(), want) <= FP64_TOL


@pytest.mark.parametrize("slices", ["1", "3"])
@pytest.mark.parametrize("tile", ["9", "10", "11"])
def test_gather_scaled_blocks(tile, slices, plans):
    """Complex contractions are two k blocks per GEMM, one of them negated;
    indexed ones a block per matching pair, scaled by the entries' factors."""
    from tests.test_gpu_complex import _case
    plans.setenv("TBLIS_HIP_PANEL_TILE", tile)
    plans.setenv("TBLIS_HIP_KSPLIT", slices)
    rng = np.random.default_rng(72000 + int(tile) * 10 + int(slices))
    _case(rng, "aebf", "fjei", "aibj", dict(a=9, b=7, e=5, f=6, i=4, j=11), torch.complex128, 0.5 - 0.25j, 1.0,
          conj_B=True)
    assert T.last_tile() == int(tile)
    d = [torch.rand(6, 35, 21, dtype=torch.float64, device=DEV) - 0.5 for _ in range(2)]
    fa, fb = [0.5, -1.0, 2.0, 1.0, 0.25, 3.0], [1.0, 1.5, -0.5, 1.0, 2.0, -1.0]
    A = T.Indexed([x for x in d[0]], [(i,) for i in range(6)], [8], fa)
    B = T.Indexed([x for x in d[1]], [(i + 1,) for i in range(6)], [8], fb)
    c = torch.zeros(35, 35, dtype=torch.float64, device=DEV)
    T.indexed_mult(1.0, A, "aef", B, "bef", 0.0, T.Indexed([c], [()], []), "ab")
    torch.cuda.synchronize()
    want = sum(fa[i + 1] * fb[i] * (d[0][i + 1].cpu() @ d[1][i].cpu().T) for i in range(5))
    assert rel_fro(c.cpu().numpy(), want.numpy()) <= FP64_TOL


@pytest.mark.parametrize("m,n,k", [(32, 32, 8192), (1, 1, 5000), (3, 65, 4097), (64, 32768, 32),
                                   (60, 36001, 63), (513, 600, 70)])
def test_gather_chosen_by_shape(m, n, k, plans):
    """Long sums into few results and short sums into many take the gather
    tiles without a knob, and TBLIS_HIP_DIRECT=0 packs as before."""
    g = torch.Generator(device=DEV).manual_seed(73000 + k)
    A = torch.rand(k, m, dtype=torch.float64, device=DEV, generator=g).t() - 0.5
    B = torch.rand(n, k, dtype=torch.float64, device=DEV, generator=g).t() - 0.5
    C0 = torch.rand(n, m, dtype=torch.float64, device=DEV, generator=g).t()
    want = 0.5 * (A.cpu().numpy() @ B.cpu().numpy()) + 2.0 * C0.cpu().numpy()
    for direct, both in (("1", True), ("0", False)):
        plans.setenv("TBLIS_HIP_DIRECT", direct)
        T.lib().tblis_hip_clear_plan_cache()
        C = C0.clone()
        T.mult(0.5, A, "ak", B, "kb", 2.0, C, "ab")
        torch.cuda.synchronize()
        assert (T.last_tile() >= 9) == both
        assert rel_fro(C.cpu().numpy(), want) <= FP64_TOL


def test_sliced_call_in_a_graph(plans):
    """A plan cut along k is two launches and a workspace: captured once, and
    every replay agrees with the eager call while eager calls run between."""
    g = torch.Generator(device=DEV).manual_seed(74000)
    A = torch.rand(20000, 24, dtype=torch.float64, device=DEV, generator=g) - 0.5
    B = torch.rand(20000, 40, dtype=torch.float64, device=DEV, generator=g) - 0.5
    want = A.cpu().numpy().T @ B.cpu().numpy()
    C = torch.zeros(24, 40, dtype=torch.float64, device=DEV)
    D = torch.zeros(24, 40, dtype=torch.float64, device=DEV)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    T.set_stream(side.cuda_stream)
    try:
        T.mult(1.0, A, "km", B, "kn", 0.0, C, "mn")
        assert T.last_tile() >= 9
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            T.mult(1.0, A, "km", B, "kn", 0.0, C, "mn")
    finally:
        T.set_stream(0)
    for _ in range(4):
        C.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert rel_fro(C.cpu().numpy(), want) <= FP64_TOL
        T.mult(2.0, A, "km", B, "kn", 0.0, D, "mn")
        torch.cuda.synchronize()
        assert rel_fro(D.cpu().numpy(), 2.0 * want) <= FP64_TOL


def _f32_case(m, n, k, ra, rb, at, g, alpha=1.25, beta=-0.5):
    """C = alpha A B + beta C on tensors `at` floats past a 16-byte boundary.
    Returns the error's norm over the result's; over |alpha| |A| |B| + |beta|
    |C| where the result is a single entry, whose two terms may cancel."""

    def tensor(shape, row_major):
        v = (torch.rand(at + shape[0] * shape[1], device=DEV, generator=g) - 0.5)[at:]
        return v.view(shape) if row_major else v.view(shape[1], shape[0]).t()

    A, B, C = tensor((m, k), ra), tensor((k, n), rb), tensor((m, n), True)
    a, b, c = (x.double().cpu() for x in (A, B, C))
    want, size = alpha * (a @ b) + beta * c, abs(alpha) * (a.abs() @ b.abs()) + abs(beta) * c.abs()
    if m * n > 1:
        size = want
    T.mult(alpha, A, "ak", B, "kb", beta, C, "ab")
    torch.cuda.synchronize()
    return ((C.double().cpu() - want).norm() / size.norm()).item()


@pytest.mark.parametrize("at", [0, 1])
@pytest.mark.parametrize("slices", ["1", "3"])
@pytest.mark.parametrize("tile", ["6", "7"])
def test_gather_split_bf16(tile, slices, at, plans):
    """The split-BF16 gather tiles: lanes along rows or along k on either
    side, rows in aligned eights or not, k below, at and past a stage, one row
    or column, edges of tiles.  Bar: 1e-6, the bound of every split-BF16 path
    (three BF16 terms hold a float; what the sums of at most 1100 products in
    float lose stays under 16 units of 2^-24)."""
    plans.setenv("TBLIS_HIP_PANEL_TILE", tile)
    plans.setenv("TBLIS_HIP_KSPLIT", slices)
    g = torch.Generator(device=DEV).manual_seed(76000 + int(tile) * 10 + int(slices) + at)
    for m, n, k in [(1, 1, 1), (1, 65, 17), (64, 64, 32), (128, 136, 16), (129, 127, 47), (65, 63, 33), (200, 8, 80),
                    (8, 264, 1100), (130, 62, 31)]:
        for ra in (False, True):
            for rb in (False, True):
                assert _f32_case(m, n, k, ra, rb, at, g) <= 1e-6, (m, n, k, ra, rb)
                assert T.last_tile() == int(tile)
    # k of two dimensions, odd extents, an operand with no unit stride along
    # its rows or k in the order of C; beta = 0 over NaN
    for A, B, C in [("eafb", "jefi", "iabj"), ("aebf", "fjei", "aibj"), ("feba", "ijfe", "baji")]:
        ext = dict(a=7, b=9, e=5, f=13, i=3, j=11)
        x, y = (torch.rand([ext[d] for d in s], device=DEV, generator=g) - 0.5 for s in (A, B))
        c = torch.full([ext[d] for d in C], float("nan"), device=DEV)
        T.mult(1.0, x, A, y, B, 0.0, c, C)
        torch.cuda.synchronize()
        want = np.einsum(f"{A},{B}->{C}", x.double().cpu().numpy(), y.double().cpu().numpy())
        assert rel_fro(c.double().cpu().numpy(), want) <= 1e-6, (A, B, C)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_orders_of_the_general_path(dtype, plans):
    """Every order of the labels in both operands gives what packing gives,
    whichever way the gather tiles walk them (the sums over e, f are long
    enough for them to reorder rows and k)."""
    import itertools
    ext = dict(a=18, b=7, e=21, f=14, i=5, j=19)
    g = torch.Generator(device=DEV).manual_seed(77000)
    tol = 1e-12 if dtype == torch.float64 else 1e-6
    for n, (A, B) in enumerate(itertools.product(list(itertools.permutations("abef"))[::3],
                                                 list(itertools.permutations("efij"))[::5])):
        C = ["abij", "jiba", "iabj", "bjai"][n % 4]
        x, y = (torch.rand([ext[d] for d in s], dtype=dtype, device=DEV, generator=g) - 0.5 for s in (A, B))
        out = []
        for direct in ("1", "0"):
            plans.setenv("TBLIS_HIP_DIRECT", direct)
            T.lib().tblis_hip_clear_plan_cache()
            c = torch.ones([ext[d] for d in C], dtype=dtype, device=DEV)
            T.mult(1.0, x, "".join(A), y, "".join(B), 0.5, c, C)
            torch.cuda.synchronize()
            out.append(c.double().cpu().numpy())
        assert rel_fro(out[0], out[1]) <= tol, (A, B, C)


@pytest.mark.parametrize("m,n,k,gather", [(64, 64, 64, True), (1296, 1296, 1296, True), (32, 32, 8192, True),
                                          (4096, 4096, 2048, False)])
def test_split_bf16_chosen_by_shape(m, n, k, gather, plans):
    """The split-BF16 gather tiles run without a knob; large operands in even
    rounds of 256 x 128 tiles, and TBLIS_HIP_DIRECT=0, take the panel tiles."""
    g = torch.Generator(device=DEV).manual_seed(78000 + k)
    for direct in ("1", "0"):
        plans.setenv("TBLIS_HIP_DIRECT", direct)
        T.lib().tblis_hip_clear_plan_cache()
        assert _f32_case(m, n, k, False, False, 0, g) <= 1e-6
        assert (T.last_tile() >= 6) == (gather and direct == "1")


@pytest.mark.parametrize("m,n,k", [(1225, 1225, 120), (33, 4489, 225), (1025, 1023, 31), (2500, 31, 2499), (71, 5041, 35)])
def test_tiles_by_rounds(m, n, k, plans):
    """Odd extents, where whole rounds of waves choose among register-fed and
    gather tiles, on every side of the rule's line."""
    rng = np.random.default_rng(79000 + m)
    _dense_case(rng, "ak", "kb", "ab", dict(a=m, b=n, k=k), ["col"] * 3, alpha=0.5, beta=2.0)
    _dense_case(rng, "ak", "kb", "ab", dict(a=m, b=n, k=k), ["row", "col", "row"], alpha=1.0, beta=0.0)


@pytest.mark.parametrize("m,n,k", [(2304, 2304, 40), (2401, 2401, 96), (2049, 2047, 33), (2561, 2049, 1700)])
def test_split_bf16_tiles_by_rounds(m, n, k, plans):
    """Around the line between gathering and packing large operands."""
    g = torch.Generator(device=DEV).manual_seed(80000 + m)
    assert _f32_case(m, n, k, False, False, 0, g) <= 1e-6


@pytest.mark.parametrize("v", [9, 17, 30, 33])
def test_complex_split_bf16_tiles(v, plans):
    """complex64 GEMMs over the sizes where the panel tile changes."""
    from tests.test_gpu_complex import _case
    rng = np.random.default_rng(81000 + v)
    _case(rng, "abef", "efij", "abij", dict(a=v, b=v, e=3, f=7, i=v, j=v), torch.complex64, 0.5 - 0.25j, 1.0)


def _mult_turned(A, la, negA, B, lb, negB, C_, lc, negC, alpha, beta):
    """T.mult on descriptors whose dimensions in neg* run backwards (data at
    their last element, negative stride); returns the tensors as seen."""
    import ctypes
    from tblis_amd import _Desc
    descs, seen = [], []
    for x, labels, neg, s in ((A, la, negA, alpha), (B, lb, negB, 1.0), (C_, lc, negC, beta)):
        d = _Desc(x, s)
        at = x.data_ptr()
        for i, label in enumerate(labels):
            if label in neg:
                at += (x.shape[i] - 1) * x.stride(i) * x.element_size()
                d.stride[i] = -x.stride(i)
        d.d.data = ctypes.c_void_p(at)
        descs.append(d)
        seen.append(lambda x=x, labels=labels, neg=neg:
                    x.double().cpu().flip([i for i, label in enumerate(labels) if label in neg]).numpy())
    before = [s() for s in seen]
    T.lib().tblis_tensor_mult(None, None, *[y for d, labels in zip(descs, (la, lb, lc))
                                            for y in (ctypes.byref(d.d), labels.encode())])
    torch.cuda.synchronize()
    return before, seen[2]()


@pytest.mark.parametrize("dtype,tol", [(torch.float64, FP64_TOL), (torch.float32, 1e-6)])
def test_negative_strides(dtype, tol, plans):
    """Descending rows, k, both, and results, on even extents (where ascending
    operands are read in 16-byte pieces) and odd ones, against the general
    path's bar for each type."""
    g = torch.Generator(device=DEV).manual_seed(83000)
    for ext in (dict(a=64, b=66, e=8, f=16), dict(a=33, b=7, e=5, f=13), dict(a=16, b=16, e=64, f=80)):
        for la, lb in (("aef", "efb"), ("fea", "bef"), ("eaf", "ebf")):
            for negA, negB, negC in (("e", "", ""), ("ef", "", ""), ("a", "b", "a"), ("aef", "bef", ""),
                                     ("", "f", "b"), ("ef", "ef", "ab")):
                A, B, C = (torch.rand([ext[x] for x in reversed(s)], dtype=dtype, device=DEV, generator=g)
                           .permute(*reversed(range(len(s)))) - 0.5 for s in (la, lb, "ab"))
                (a, b, c), got = _mult_turned(A, la, negA, B, lb, negB, C, "ab", negC, 1.5, -0.5)
                want = 1.5 * np.einsum(f"{la},{lb}->ab", a, b) - 0.5 * c
                assert rel_fro(got, want) <= tol, (ext, la, lb, negA, negB, negC)
