"""The projections' GEMMs (proj_gemm.hip: bf16 by DMA, and split operands for
fp32 tensors and other widths) and lowrank_split (proj_lora.hip) at the edges
of their tiles, against float64 products of the same operands on the GPU.

Bound per element: the result's rounding to bf16 (8 significant bits with the
implicit one: neighbours are 2^-7 apart relative to the lower power of two,
so half of that, 2^-8 relative) plus fp32
summation over n terms, n 2^-24 sum |terms| in the worst case; the sums
round to both sides, so sqrt(n) 2^-22 sum |terms| holds with room, and the
low-rank operands enter with all 24 bits (split3.hpp) within the same bound.
fp32 results have 2^-24 in the place of 2^-8.
"""
import sys

import pytest

import glacier_attn as ga

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engines():
    assert torch.cuda.is_available(), "GPU tests need a ROCm GPU"
    made = {torch.bfloat16: ga.GpuAttentionEngine(0, ga.PREC_BF16),
            torch.float32: ga.GpuAttentionEngine(0, ga.PREC_FP32)}
    yield made
    for e in made.values():
        e.close()


@pytest.fixture(scope="module")
def engine(engines):
    return engines[torch.bfloat16]


def _problem(T, n_in, outs, rank, seed=3, w_shift=0, dtype=torch.bfloat16):
    """w_shift: elements by which each W misses its allocation's alignment."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    x = rnd(T, n_in).to(dtype)
    projs = []
    for i, o in enumerate(outs):
        w = torch.empty(o * n_in + w_shift, device="cuda", dtype=dtype)[w_shift:]
        w = w.view(o, n_in).copy_(rnd(o, n_in) * n_in ** -0.5)
        p = {"w": w, "bias": 0.1 * rnd(o), "dy": rnd(T, o).to(dtype), "scaling": 2.0}
        if i != 1:  # the second projection has no adapter
            p.update(a=rnd(n_in, rank) * n_in ** -0.5, b=0.1 * rnd(rank, o))
            p.update(grad_a=torch.zeros_like(p["a"]), grad_b=torch.zeros_like(p["b"]))
        projs.append(p)
    return x, projs


def _reference(x, projs):
    """(value, sum of |terms|) of each y and of dx, in float64."""
    x = x.double()
    ys, dx = [], [0.0, 0.0]
    for p in projs:
        w, dy = p["w"].double(), p["dy"].double()
        y, bound = x @ w.t() + p["bias"].double(), x.abs() @ w.abs().t() + p["bias"].double().abs()
        d, d_bound = dy @ w, dy.abs() @ w.abs()
        if "a" in p:
            a, b, s = p["a"].double(), p["b"].double(), p["scaling"]
            y, bound = y + s * (x @ a) @ b, bound + s * (x.abs() @ a.abs()) @ b.abs()
            d, d_bound = d + s * (dy @ b.t()) @ a.t(), d_bound + s * (dy.abs() @ b.abs().t()) @ a.abs().t()
        ys.append((y, bound))
        dx = [dx[0] + d, dx[1] + d_bound]
    return ys, tuple(dx)


def _check(got, want, terms, n, what):
    err = (got.double() - want).abs()
    bound = 2.0 ** (-8 if got.dtype == torch.bfloat16 else -24) * want.abs() + n ** 0.5 * 2.0 ** -22 * terms
    worst = float((err / bound).max())
    print(f"  {what}: worst error {worst:.2f} of its bound", flush=True)
    assert worst <= 1.0


SHAPES = [  # T, in, outs, rank
    (1, 8, (8,), 1),                       # one piece of one row
    (37, 1000, (1000, 200, 200), 5),       # reduction tails, padded term rows
    (65, 72, (264, 8), 64),                # a token past the tile, the largest rank
    (129, 136, (128, 72, 136), 17),        # a second rank tile
    (512, 3584, (3584, 512, 512), 16),
    (640, 2056, (1032, 1032), 8),
    (1290, 520, (2056, 136), 33),
    (2051, 1024, (2048, 520, 264), 16),    # taller low-rank slabs
    (4099, 256, (4104,), 12),              # 128 x 128 tiles, two to a CU, ragged in both directions
    (2051, 4088, (4088,), 24),             # 256 x 256 tiles in both directions, ragged in both
    (2051, 2040, (1032, 8), 40),           # 128 x 128 tiles two to a CU backward
]


OTHER_SHAPES = [  # the split-operand GEMM
    (torch.float32, 1, 4, (4,), 1),
    (torch.float32, 37, 100, (36, 72), 3),
    (torch.float32, 65, 1000, (1000, 200, 200), 20),
    (torch.float32, 130, 264, (516, 4), 64),
    (torch.float32, 512, 3584, (3584, 512, 512), 16),  # the larger tiles forward
    (torch.float32, 1025, 520, (2052,), 8),            # the larger tiles, ragged: forward
    (torch.float32, 1025, 2052, (520,), 8),            # and backward
    (torch.bfloat16, 37, 100, (36, 72), 3),            # rows of half 16-byte pieces
    (torch.bfloat16, 700, 1004, (3004, 12), 17),
]


def _run_and_check(eng, x, projs, rank):
    n_in = x.shape[1]
    ys = eng.proj_forward(x, projs, rank)
    dx = eng.proj_backward(x, projs, rank)
    want, want_dx = _reference(x, projs)
    for i, (y, (ref, terms)) in enumerate(zip(ys, want)):
        _check(y, ref, terms, n_in, f"y{i}")
    _check(dx, *want_dx, sum(p["w"].shape[0] for p in projs), "dx")
    xd = x.double()
    for p in projs:
        if "a" not in p:
            continue
        dl, l = p["dy"].double() @ p["b"].double().t(), xd @ p["a"].double()
        for got, ref in ((p["grad_a"], 2.0 * xd.t() @ dl), (p["grad_b"], 2.0 * l.t() @ p["dy"].double())):
            assert float((got.double() - ref).norm() / ref.norm()) <= 2e-6  # fp32 sums


@pytest.mark.parametrize("T,n_in,outs,rank", SHAPES)
def test_fused_projection_matches_float64(engine, T, n_in, outs, rank):
    print(f"[fused proj] T={T} in={n_in} outs={outs} rank={rank}", flush=True)
    sys.stdout.flush()
    _run_and_check(engine, *_problem(T, n_in, outs, rank), rank)


@pytest.mark.parametrize("dtype,T,n_in,outs,rank", OTHER_SHAPES)
def test_split_projection_matches_float64(engines, dtype, T, n_in, outs, rank):
    print(f"[split proj] {dtype} T={T} in={n_in} outs={outs} rank={rank}", flush=True)
    sys.stdout.flush()
    _run_and_check(engines[dtype], *_problem(T, n_in, outs, rank, dtype=dtype), rank)


def test_unaligned_weights_take_the_general_path(engine):
    """The DMA moves aligned 16-byte pieces; weights that are not stay with
    the general kernels and give the same products."""
    x, projs = _problem(70, 136, (72, 136), 8, w_shift=4)
    assert projs[0]["w"].data_ptr() % 16 != 0
    ys = engine.proj_forward(x, projs, 8)
    dx = engine.proj_backward(x, projs, 8)
    want, want_dx = _reference(x, projs)
    for y, (ref, terms) in zip(ys, want):
        _check(y, ref, terms, 136, "y")
    _check(dx, *want_dx, 208, "dx")


@pytest.mark.parametrize("where", ["x", "a", "b", "dy", "huge_b"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_non_finite_values_pass_through(engines, dtype, where):
    """Infinities, NaN and values past bf16's range have no split terms: the
    results hold inf and NaN exactly where float32 arithmetic does, and every
    other element is unharmed."""
    T, n_in, outs, rank = 70, 136, (72, 64), 8
    engine = engines[dtype]
    x, projs = _problem(T, n_in, outs, rank, dtype=dtype)
    p = projs[0]
    if where == "x":
        x[5, 7], x[9, 3] = float("inf"), float("nan")
    elif where == "a":
        p["a"][11, 2], p["a"][12, 3] = float("-inf"), float("nan")
    elif where == "b":
        p["b"][1, 20], p["b"][2, 21] = float("inf"), float("nan")
    elif where == "dy":
        p["dy"][6, 8] = float("inf")
    else:
        p["b"][1, 20] = 3.4e38  # rounds to infinity in bf16
        for t in (x, p["dy"]):  # and whose products stay inside float32
            t.mul_(1.0e-3)
    ys = engine.proj_forward(x, projs, rank)
    dx = engine.proj_backward(x, projs, rank)
    want, want_dx = _reference(x, projs)
    for got, (ref, terms) in zip([*ys, dx], [*want, want_dx]):
        ref32 = ref.float().to(dtype)
        assert torch.equal(torch.isnan(got), torch.isnan(ref32))
        assert torch.equal(torch.isinf(got), torch.isinf(ref32))
        ok = torch.isfinite(ref32) & torch.isfinite(terms)
        if ok.any():
            _check(got[ok], ref[ok], terms[ok], n_in, where)


@pytest.mark.parametrize("T,n_in,outs,rank", [(201, 896, (896, 128), 8), (1100, 1024, (2048, 520), 16)])
@pytest.mark.parametrize("where", ["x", "w", "a"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_small_values_keep_their_bits(engines, dtype, where, T, n_in, outs, rank):
    """Operands down to 2^-118, whose last bits three bf16 terms do not reach
    (split3.hpp): fp32 results stay within 2e-6 of float64 in the 2-norm (fp32
    sums, the gate of the adapters' gradients), bf16 ones within 2^-8.  With
    "a" only the low-rank product is left, on activations of about 2^-120 in
    fp32 and, to show in bf16 results, 2^-130 in bf16 (19 bits in themselves)."""
    print(f"[small values] {dtype} {where} T={T} in={n_in} outs={outs} rank={rank}", flush=True)
    x, projs = _problem(T, n_in, outs, rank, dtype=dtype)
    for p in projs:
        p["bias"] = None
    if where == "a":
        x.mul_(2.0 ** -60)
        for p in projs:
            p["w"].zero_()
        projs[0]["a"].mul_(2.0 ** (-60 if dtype == torch.float32 else -70))
        projs[0]["b"].mul_(2.0 ** 30)
    else:
        for t in [x, *[p["dy"] for p in projs]] if where == "x" else [p["w"] for p in projs]:
            t.mul_(2.0 ** -118)
    if where == "w":
        projs[0]["a"].mul_(2.0 ** -118)
    p = projs[0]
    ys = engines[dtype].proj_forward(x, projs, rank)
    dx = engines[dtype].proj_backward(x, projs, rank)
    xd, dy = x.double(), p["dy"].double()
    low = xd @ p["a"].double()
    y = xd @ p["w"].double().t() + 2.0 * low @ p["b"].double()
    want_dx = sum(q["dy"].double() @ q["w"].double() for q in projs)
    want_dx = want_dx + 2.0 * (dy @ p["b"].double().t()) @ p["a"].double().t()
    gate = 2e-6 if dtype == torch.float32 else 2.0 ** -8
    for got, want, within in ((ys[0], y, gate), (dx, want_dx, gate),
                              (p["grad_b"], 2.0 * low.t() @ dy, gate if where == "a" else 2e-6)):
        if float(want.abs().max()) < 2.0 ** -118:
            continue  # results of few bits themselves
        scale = 2.0 ** 100  # squares inside float64 either way; norms of small numbers stay normal
        err = float(((got.double() - want) * scale).norm() / (want * scale).norm())
        print(f"  {err:.2e} of {within:.2e}", flush=True)
        assert err <= within


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [1024, 1028])  # both GEMMs in bf16
def test_outputs_in_the_place_of_inputs(engines, dtype, n):
    """dx in a dY's memory, and y in x's (out == in), are what they are beside
    them: every workgroup reads its operands before anything replaces them."""
    print(f"[in place] {dtype} n={n}", flush=True)
    T, rank = 300, 8
    x, projs = _problem(T, n, (n, 8, n), rank, dtype=dtype)
    eng = engines[dtype]
    dx = eng.proj_backward(x, projs, rank).clone()
    ys = [y.clone() for y in eng.proj_forward(x, projs, rank)]
    place = projs[2]["dy"]
    assert torch.equal(eng.proj_backward(x, projs, rank, dx=place), dx)
    x_in, projs[0]["y"] = x, x
    for got, want in zip(eng.proj_forward(x_in, projs, rank), ys):
        assert torch.equal(got, want)


# how far fp32 MFMAs and a reduction split over workgroups were from float64 at
# these sizes (2-norm), and a tenth for the draw
@pytest.mark.parametrize("dtype,T,n_in,outs,rank,y_gate,dx_gate,grad_gate", [
    (torch.float32, 152, 3584, (3584, 512, 512), 32, 8.0e-7, 9.1e-7, 2.1e-7),
    (torch.float32, 538, 896, (896, 128, 128), 64, 3.7e-7, 4.7e-7, 2.3e-7),
    (torch.bfloat16, 19, 4096, (4096, 1024, 1024), 64, None, None, 1.7e-7)])
def test_split_sums_are_as_exact_as_fp32_ones(engines, dtype, T, n_in, outs, rank, y_gate, dx_gate,
                                              grad_gate):
    """Splitting an fp32 operand adds sums, and each rounds: the small products
    have a sum of their own, so that the result is no further from float64."""
    print(f"[split sums] {dtype} T={T} in={n_in} outs={outs} rank={rank}", flush=True)
    x, projs = _problem(T, n_in, outs, rank, dtype=dtype)
    for p in projs:
        p["bias"] *= 0.0
    ys, dx = engines[dtype].proj_forward(x, projs, rank), engines[dtype].proj_backward(x, projs, rank)
    want, want_dx = _reference(x, projs)
    err = lambda got, ref: float((got.double() - ref).norm() / ref.norm())  # noqa: E731
    if y_gate is not None:
        assert err(ys[0], want[0][0]) <= y_gate
        assert err(dx, want_dx[0]) <= dx_gate
    xd = x.double()
    for p in projs:
        if "a" not in p:
            continue
        dl, low = p["dy"].double() @ p["b"].double().t(), xd @ p["a"].double()
        for name, ref in (("grad_a", 2.0 * xd.t() @ dl), ("grad_b", 2.0 * low.t() @ p["dy"].double())):
            print(f"  {name} {err(p[name], ref):.2e} of {grad_gate:.1e}", flush=True)
            assert err(p[name], ref) <= grad_gate


# one term for bf16 operands of the general GEMM: rows of 4, rows that end 4
# before a 16-byte piece, one row, the larger tiles in both directions
ODD_WIDTHS = [  # T, in, outs, rank
    (1, 4, (4,), 1), (70, 12, (4, 36), 3), (33, 4, (12,), 2), (1, 12, (12, 8), 2),
    (65, 268, (132, 8), 16), (1025, 2052, (2052,), 16)]


@pytest.mark.parametrize("T,n_in,outs,rank", ODD_WIDTHS)
def test_odd_bf16_widths_match_float64(engine, T, n_in, outs, rank):
    print(f"[odd widths] T={T} in={n_in} outs={outs} rank={rank}", flush=True)
    _run_and_check(engine, *_problem(T, n_in, outs, rank), rank)


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_non_finite_row_ends_stay_in_their_rows(engine, value):
    """Loads past a row's end repeat its last elements: where those are not
    finite, the zeros of the other operand have to meet zeros."""
    T, n_in, outs, rank = 70, 100, (36, 72), 3
    x, projs = _problem(T, n_in, outs, rank)
    x[5, n_in - 1] = value
    projs[0]["dy"][6, outs[0] - 1] = value
    projs[1]["w"][7, n_in - 2] = value
    ys, dx = engine.proj_forward(x, projs, rank), engine.proj_backward(x, projs, rank)
    want, want_dx = _reference(x, projs)
    for got, (ref, terms) in zip([*ys, dx], [*want, want_dx]):
        ref = ref.float().to(got.dtype)
        assert torch.equal(torch.isnan(got), torch.isnan(ref))
        assert torch.equal(torch.isinf(got), torch.isinf(ref))
        ok = torch.isfinite(ref)
        _check(got[ok], ref[ok], terms[ok], n_in, "finite")


# lowrank_split: rank tiles over its workgroups (one, two and four to a workgroup,
# the last one partial or absent), then slabs of two and of four row blocks
RANKS = [  # T, outs, rank
    (37, (136,), 17), (37, (136,), 64), (1100, (136,), 40), (1100, (136,), 64), (1900, (136,), 33),
    (1401, (136, 8, 72), 8), (1401, (136, 8, 72), 20), (1401, (136, 8, 72), 40), (1401, (136, 8, 72), 64),
    (2107, (136, 8, 72), 16), (2107, (136, 8, 72), 20)]
RANK_WIDTHS = [(torch.bfloat16, 264), (torch.bfloat16, 268), (torch.float32, 264)]


@pytest.mark.parametrize("dtype,n_in", RANK_WIDTHS)
@pytest.mark.parametrize("T,outs,rank", RANKS)
def test_low_rank_shapes_match_float64(engines, dtype, n_in, T, outs, rank):
    print(f"[low rank] {dtype} T={T} in={n_in} outs={outs} rank={rank}", flush=True)
    _run_and_check(engines[dtype], *_problem(T, n_in, outs, rank, dtype=dtype), rank)


@pytest.mark.parametrize("dtype,T,n_in,outs,where", [
    (torch.bfloat16, 2051, 4088, (4088,), "b"), (torch.bfloat16, 2051, 2040, (1032,), "a"),
    (torch.float32, 1025, 520, (2052,), "x"), (torch.float32, 1025, 2052, (520,), "dy")])
def test_non_finite_values_in_large_tiles(engines, dtype, T, n_in, outs, where):
    """As in the smallest tiles: the low-rank product of the whole call, or the
    tile that holds the value, on fp32 products."""
    print(f"[large non-finite] {dtype} T={T} in={n_in} outs={outs} {where}", flush=True)
    rank = 8
    x, projs = _problem(T, n_in, outs, rank, dtype=dtype)
    p = projs[0]
    place = {"x": x, "dy": p["dy"], "a": p["a"], "b": p["b"]}[where]
    place[place.shape[0] - 2, place.shape[1] - 3] = float("inf")
    ys, dx = engines[dtype].proj_forward(x, projs, rank), engines[dtype].proj_backward(x, projs, rank)
    want, want_dx = _reference(x, projs)
    for got, (ref, terms) in zip([*ys, dx], [*want, want_dx]):
        ref32 = ref.float().to(dtype)
        assert torch.equal(torch.isnan(got), torch.isnan(ref32))
        assert torch.equal(torch.isinf(got), torch.isinf(ref32))
        ok = torch.isfinite(ref32) & torch.isfinite(terms)
        if ok.any():
            _check(got[ok], ref[ok], terms[ok], max(n_in, outs[0]), where)
