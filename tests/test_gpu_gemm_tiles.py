"""The GEMMs of csrc/dit_gemm.hip in every tile shape, data type and epilogue,
each shape asked for by its index (the dispatch's estimate reaches only some of
them at the sizes of the block tests), against float64 products.

Sizes end inside a tile in both directions and, over the values of K, inside a
stage (64 bf16 or 32 fp32 values), with one to seven stages: fewer than a tile
has buffers, as many, and more.

Bounds, per output and from its own terms (S = sum |a w|): a product of split
operands keeps 2^-22 of each operand and drops at most 2^-22 (lo lo), and what
small values lose is at most 2^-22 of the output; sums of 16 products a step are
rounded to fp32, so (3 + 1) 2^-22 S + (K / 16 + 4) 2^-24 S. bf16 operands are exact
and rounded once more on the store, 2^-8 of the result. The epilogues scale that by their
derivatives (|silu'| < 1.1) and add their own roundings."""

import ctypes

import numpy as np
import pytest

import awa_hip as A

pytestmark = pytest.mark.gpu

STORE, GATE, SWIGLU = 0, 1, 2
TILES = [(256, 256), (256, 192), (128, 256), (128, 192), (128, 192), (64, 128), (64, 64)]


class GemmStep(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int) for n in ("split", "tile", "epilogue", "n", "k")] + \
        [(n, ctypes.c_int * 2) for n in ("rows", "twice")] + \
        [(n, ctypes.c_void_p * 2) for n in ("a", "w", "w2", "residual", "bias", "gate", "out")]


def to_device(x, es):
    x = np.ascontiguousarray(x, np.float32)
    buf = A.DeviceBuffer(x.size * es)
    buf.upload(A.f32_to_bf16_bits(x) if es == 2 else x)
    return buf


def from_device(buf, shape, es):
    raw = buf.download((int(np.prod(shape)),), np.uint16 if es == 2 else np.float32)
    return (A.bf16_bits_to_f32(raw) if es == 2 else raw).reshape(shape)


def operands(rng, rows, n, k, epilogue, es):
    """One branch's operands as the kernel holds them."""
    rounded = (lambda x: A.bf16_bits_to_f32(A.f32_to_bf16_bits(x)).reshape(x.shape)) if es == 2 else (lambda x: x)
    normal = lambda *s, sd=1.0: (rng.standard_normal(s) * sd).astype(np.float32)
    half = n // 2 if epilogue == SWIGLU else n
    op = {"a": rounded(normal(rows, k)), "w": rounded(normal(half, k, sd=0.1))}
    if epilogue == SWIGLU:
        op["w2"] = rounded(normal(half, k, sd=0.1))
    if epilogue == GATE:
        op.update(residual=rounded(normal(rows, n)), bias=normal(n), gate=normal(n))
    return op


def run(split, tile, epilogue, n, k, branches, off_16=False):
    """off_16: the weights one element into their allocations (split only)."""
    es = 4 if split else 2
    step = GemmStep(split=split, tile=tile, epilogue=epilogue, n=n, k=k)
    width = n // 2 if epilogue == SWIGLU else n
    keep, outs = [], []
    for br, op in enumerate(branches):
        rows = op["a"].shape[0]
        step.rows[br] = rows
        step.twice[br] = br if epilogue == GATE else 0
        for name, x in op.items():
            moved = off_16 and name in ("w", "w2")
            keep.append(to_device(np.append(np.float32(0), x) if moved else x, 4 if name in ("bias", "gate") else es))
            getattr(step, name)[br] = keep[-1].ptr + (es if moved else 0)
        outs.append(A.DeviceBuffer(rows * width * es))
        step.out[br] = outs[-1].ptr
    A.check(A.lib().awa_gemm_step_run(ctypes.byref(step), None), "awa_gemm_step_run")
    A.synchronize()
    return [from_device(o, (op["a"].shape[0], width), es) for o, op in zip(outs, branches)], step.tile


def expected(op, epilogue, twice, es):
    """The outputs in float64 and the bound of each."""
    k = op["a"].shape[1]
    f = {name: x.astype(np.float64) for name, x in op.items()}

    def product(w):
        with np.errstate(invalid="ignore"):
            y = f["a"] @ w.T
            s = np.abs(np.where(np.isfinite(f["a"]), f["a"], 0)) @ np.abs(np.where(np.isfinite(w), w, 0)).T
        return y, s * ((4 * 2.0 ** -22 if es == 4 else 0) + (k / 16 + 4) * 2.0 ** -24)

    y, e = product(f["w"])
    with np.errstate(invalid="ignore", over="ignore"):
        if epilogue == GATE:
            own = np.abs((y + f["bias"]) * f["gate"]) + np.abs(f["residual"])
            y = (y + f["bias"]) * f["gate"] + f["residual"]
            y, e = (1 + twice) * y, (1 + twice) * (e * np.abs(f["gate"]) + own * 2.0 ** -22)
        if epilogue == SWIGLU:
            z, ez = product(f["w2"])
            silu = y / (1 + np.exp(-y))
            y, e = silu * z, 1.1 * e * (np.abs(z) + ez) + np.abs(silu) * ez
            e = e + np.abs(y) * (2.0 ** -21 if es == 4 else 2.0 ** -17)
        return y, e + (np.abs(y) * 2.0 ** -8 if es == 2 else 0)


def compare(got, op, epilogue, twice, es, what):
    ref, bound = expected(op, epilogue, twice, es)
    finite = np.isfinite(ref)
    assert np.array_equal(np.isnan(got), np.isnan(ref)), what
    assert np.array_equal(got[np.isinf(ref)].astype(np.float64), ref[np.isinf(ref)]), what
    worst = np.max(np.abs(got[finite].astype(np.float64) - ref[finite]) / (bound[finite] + 1e-37), initial=0.0)
    assert worst <= 1.0, f"{what}: {worst:.3g} of the bound"
    return worst


def size_of(tile, epilogue):
    bm, bn = TILES[tile]
    return bm + 33, (2 * (bn // 2 + 24) if epilogue == SWIGLU else bn + 40)


@pytest.mark.parametrize("epilogue", [STORE, GATE, SWIGLU])
@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("split", [0, 1])
def test_every_tile_shape(gpu, split, tile, epilogue):
    print(f"case GEMM split={split} tile={tile} epilogue={epilogue}", flush=True)
    es, stage = (4, 32) if split else (2, 64)
    rng = np.random.default_rng(100 * tile + 10 * epilogue + split)
    rows, n = size_of(tile, epilogue)
    worst = 0.0
    for stages in range(1, 8):
        for k in (stage * stages, stage * stages - 24):
            # A text problem of its own, of one row, or none.
            text = {0: 70, 1: 1, 2: 0}[stages % 3]
            branches = [operands(rng, m, n, k, epilogue, es) for m in (rows, text) if m]
            got, _ = run(split, tile, epilogue, n, k, branches)
            for br, (a, op) in enumerate(zip(got, branches)):
                worst = max(worst, compare(a, op, epilogue, br if epilogue == GATE else 0, es,
                                           f"k={k} text={text} branch={br}"))
    print(f"  worst {worst:.3g} of the bound", flush=True)


@pytest.mark.parametrize("kind", ["some", "all"])
@pytest.mark.parametrize("epilogue", [STORE, GATE, SWIGLU])
@pytest.mark.parametrize("tile", range(len(TILES)))
def test_outputs_that_planes_cannot_give(gpu, tile, epilogue, kind):
    """Split GEMMs whose rows hold infinities, NaN and values that vanish as
    planes; some outputs (a few of 32 rows and whole rows of them), and all.
    Weights on 16-byte addresses and off them."""
    print(f"case GEMM marked outputs tile={tile} epilogue={epilogue} {kind}", flush=True)
    rng = np.random.default_rng(7 + 10 * tile + epilogue)
    rows, n = size_of(tile, epilogue)
    for k in (96, 232):
        branches = [operands(rng, m, n, k, epilogue, 4) for m in (rows, 70)]
        for op in branches:
            a, w = op["a"], op["w"]
            if kind == "all":
                # One huge value a row that meets zeros.
                a[:, 10] *= np.float32(2.0 ** 36)
                w[:, 10] = 0
                if "w2" in op:
                    op["w2"][:, 10] = 0
                continue
            a[:, 9] *= np.float32(2.0 ** -60)
            w[20] = 0
            w[20, 9] = 2.0 ** 60                # nothing but the vanished value
            w[21, 9] = np.inf                   # an infinity meets it
            w[len(w) - 1, k - 1] = -np.inf
            w[7, 2] = np.nan
            op.get("w2", w)[30, 5] = np.inf
            a[5, 3] = np.inf
            a[len(a) - 1, 0] = np.nan
            a[40] *= np.float32(2.0 ** 100)     # a row of another scale
            if epilogue == SWIGLU:
                w[20, 9] = 2.0 ** 58            # silu of a moderate value
                a[40] *= np.float32(2.0 ** -100)
        got, _ = run(1, tile, epilogue, n, k, branches, off_16=k == 232)
        for br, (x, op) in enumerate(zip(got, branches)):
            compare(x, op, epilogue, br if epilogue == GATE else 0, 4, f"k={k} branch={br}")


@pytest.mark.parametrize("split", [0, 1])
def test_the_estimate_takes_a_tile(gpu, split):
    """Without an index the estimate's tile runs, and large problems take
    larger tiles than small ones."""
    rng = np.random.default_rng(3)
    taken = []
    for rows, n, k in ((40, 64, 64), (1300, 2048, 2560)):
        op = operands(rng, rows, n, k, STORE, 4 if split else 2)
        got, tile = run(split, -1, STORE, n, k, [op])
        compare(got[0], op, STORE, 0, 4 if split else 2, f"rows={rows}")
        taken.append(TILES[tile][0] * TILES[tile][1])
    assert taken[0] < taken[1]
