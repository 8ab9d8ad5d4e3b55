"""DiT blocks on the GEMMs of csrc/dit_gemm.hip (bf16, and fp32 as two fp16
planes a row) against the oracle block, at sizes off every tile: rows and
columns that end inside a tile, widths that are no multiple of the 32 (fp32)
or 64 (bf16) values of a stage, one text token.

Tolerance, max|err| / max|ref|: the split keeps 22 bits and the sign of each
operand (2^-22 of a value, two operands a product) and sums in fp32; over K
random terms both errors grow like the result, so the fp32 block's bound of
1e-5 stands as it does for fp32 products. bf16 blocks: the bf16 budget, 2e-2.
"""

import numpy as np
import pytest

import awa_hip as A
import oracle as O
from awa_cases import geometry
from test_dit_block_oracle import EPS, HEAD_DIM
from test_gpu_dit_block import DeviceBranch, download_act, upload_act

pytestmark = pytest.mark.gpu


def weights(rng, heads, hidden, mlp):
    hd = heads * HEAD_DIM
    n = lambda *s, sd=0.05: (rng.standard_normal(s) * sd).astype(np.float32)
    return O.DitBranchWeights(qkv=n(3 * hd, hidden), proj_out=n(hidden, hd), proj_out_bias=n(hidden, sd=0.1),
                              mlp_gate=n(mlp, hidden), mlp_in=n(mlp, hidden), mlp_out=n(hidden, mlp),
                              norm_q=rng.uniform(0.5, 1.5, HEAD_DIM).astype(np.float32),
                              norm_k=rng.uniform(0.5, 1.5, HEAD_DIM).astype(np.float32), ada=n(6, hidden, sd=0.5))


def inputs(seed, grid, text, heads, hidden, mlp):
    rng = np.random.default_rng(seed)
    g = geometry(grid + (2, 8, 8, text), False)
    n = lambda *s: rng.standard_normal(s).astype(np.float32)
    return g, n(g.source_tokens, hidden), n(text, hidden), n(hidden * 6), weights(rng, heads, hidden, mlp), \
        weights(rng, heads, hidden, mlp)


def run(g, video, text, emb, wv, wt, heads, hidden, mlp, last=False, es=4, misaligned=False):
    precision = A.COMPUTE_F32 if es == 4 else A.COMPUTE_BF16
    blk = A.DitBlock(*g.args, g.text_tokens, g.shifted, heads, HEAD_DIM, hidden, mlp, last, precision, EPS)
    dv, dt = DeviceBranch(wv, es), DeviceBranch(wt, es, adjacent_mlp=True)
    if misaligned:
        # The video branch's mlp_out one element into its allocation.
        off = A.DeviceBuffer((wv.mlp_out.size + 8) * es)
        w = np.concatenate([np.zeros(1, np.float32), wv.mlp_out.reshape(-1), np.zeros(7, np.float32)])
        off.upload(A.f32_to_bf16_bits(w) if es == 2 else w)
        dv.struct.mlp_out = off.ptr + es
    bv, bt, be = upload_act(video, es), upload_act(text, es), upload_act(emb, es)
    ov, ot = A.DeviceBuffer(video.size * es), A.DeviceBuffer(text.size * es)
    blk.forward(dv.struct, dt.struct, bv.ptr, bt.ptr, be.ptr, ov.ptr, ot.ptr)
    A.synchronize()
    out = download_act(ov, video.shape, es), download_act(ot, text.shape, es)
    blk.destroy()
    return out


def off(a, b):
    return float(np.max(np.abs(a.astype(np.float64) - b)) / np.max(np.abs(b)))


@pytest.mark.parametrize("es", [4, 2])
@pytest.mark.parametrize("grid,text,heads,hidden,mlp,last", [
    ((3, 16, 16), 64, 2, 256, 384, False),   # whole tiles and stages
    ((5, 13, 13), 1, 1, 264, 392, False),    # 845 rows; widths 8 over a stage; one text token
    ((4, 16, 17), 100, 3, 248, 712, True),   # hidden short of a stage; last block
    ((1, 9, 11), 70, 1, 8, 16, False),       # 99 rows; bf16 rows of less than one stage
    ((9, 20, 24), 65, 8, 1024, 2760, False), # many tiles of the larger shapes, the last ones short
])
def test_block_matches_oracle(gpu, grid, text, heads, hidden, mlp, last, es):
    print(f"case block {grid} text={text} heads={heads} hidden={hidden} mlp={mlp} last={last} es={es}", flush=True)
    g, video, txt, emb, wv, wt = inputs(31 + hidden, grid, text, heads, hidden, mlp)
    got = run(g, video, txt, emb, wv, wt, heads, hidden, mlp, last, es)
    ref = O.dit_block(g, video, txt, emb, wv, wt, heads, HEAD_DIM, EPS, last, bf16=es == 2)
    errs = [off(a, b) for a, b in zip(got, ref)]
    print(f"  rel err video {errs[0]:.3g} text {errs[1]:.3g}", flush=True)
    assert max(errs) <= (1e-5 if es == 4 else 2e-2)


@pytest.mark.parametrize("es", [4, 2])
def test_block_takes_weights_off_16_bytes(gpu, es):
    """A weight at an address that no 16-byte load takes gives the values of
    the aligned one (fp32: the same planes and so the same bits; bf16: the
    library's GEMM, within the bf16 budget)."""
    print(f"case block misaligned weight es={es}", flush=True)
    grid, heads, hidden, mlp = (3, 16, 16), 2, 256, 384
    args = (*inputs(9, grid, 8, heads, hidden, mlp), heads, hidden, mlp)
    whole, moved = run(*args, es=es), run(*args, es=es, misaligned=True)
    for a, b in zip(whole, moved):
        assert np.array_equal(a, b) if es == 4 else off(a, b) <= 2e-2


def test_split_block_rows_of_any_scale(gpu):
    """Rows of mlp_out scaled by 2^-60 .. 2^60 (exact): every output column
    keeps the accuracy of its own scale."""
    print("case split block row scales", flush=True)
    grid, heads, hidden, mlp = (3, 16, 16), 2, 256, 384
    g, video, txt, emb, wv, wt = inputs(5, grid, 8, heads, hidden, mlp)
    scale = np.exp2(np.linspace(-60, 60, hidden).round()).astype(np.float32)
    for w in (wv, wt):
        w.mlp_out = w.mlp_out * scale[:, None]
    got = run(g, video, txt, emb, wv, wt, heads, hidden, mlp)
    ref = O.dit_block(g, video, txt, emb, wv, wt, heads, HEAD_DIM, EPS, False)
    for a, b in zip(got, ref):
        err = np.max(np.abs(a.astype(np.float64) - b), 0) / np.max(np.abs(b), 0)
        assert np.max(err) <= 1e-5


def test_split_block_infinite_and_nan_weights(gpu):
    """An infinite weight of mlp_out makes its output column infinite with
    the sign of the product, a NaN makes its column NaN; the others keep
    their values."""
    print("case split block inf nan", flush=True)
    grid, heads, hidden, mlp = (3, 16, 16), 2, 256, 384
    g, video, txt, emb, wv, wt = inputs(6, grid, 8, heads, hidden, mlp)
    clean = O.dit_block(g, video, txt, emb, wv, wt, heads, HEAD_DIM, EPS, False)
    for w in (wv, wt):
        w.mlp_out[37, 11] = np.inf
        w.mlp_out[200, 5] = -np.inf
        w.mlp_out[129, 383] = np.nan
    got = run(g, video, txt, emb, wv, wt, heads, hidden, mlp)
    with np.errstate(invalid="ignore"):
        ref = O.dit_block(g, video, txt, emb, wv, wt, heads, HEAD_DIM, EPS, False)
    keep = [c for c in range(hidden) if c not in (37, 129, 200)]
    for a, b, c in zip(got, ref, clean):
        assert np.all(np.isnan(a[:, 129]))
        for col in (37, 200):
            assert np.array_equal(a[:, col].astype(np.float64), b[:, col])
        assert off(a[:, keep], c[:, keep]) <= 1e-5


def test_split_block_infinite_hidden_value(gpu):
    """An infinite weight of mlp_in makes one hidden value of every row
    infinite (the SwiGLU epilogue), and with it every output, with the sign
    that value and its mlp_out weight give."""
    print("case split block infinite hidden value", flush=True)
    grid, heads, hidden, mlp = (3, 16, 16), 2, 256, 384
    g, video, txt, emb, wv, wt = inputs(8, grid, 8, heads, hidden, mlp)
    for w in (wv, wt):
        w.mlp_in[5, 7] = np.inf
    got = run(g, video, txt, emb, wv, wt, heads, hidden, mlp)
    with np.errstate(invalid="ignore"):
        ref = O.dit_block(g, video, txt, emb, wv, wt, heads, HEAD_DIM, EPS, False)
    for a, b in zip(got, ref):
        assert np.all(np.isinf(b))
        assert np.array_equal(a.astype(np.float64), b)


def scaled_case(kind, seed=12):
    """Block inputs whose GEMM rows hold values of very different size. fp32
    products keep every one of them; the expected block is the oracle's on the
    same numbers."""
    grid, heads, hidden, mlp = (3, 16, 16), 2, 256, 384
    g, video, txt, emb, wv, wt = inputs(seed, grid, 8, heads, hidden, mlp)
    for w in (wv, wt):
        if kind[0] == "features":
            # Four hidden features larger or smaller by 2^p, undone by mlp_out.
            w.mlp_in[[3, 100, 222, 383]] *= np.float32(2.0 ** kind[1])
            w.mlp_out[:, [3, 100, 222, 383]] *= np.float32(2.0 ** -kind[1])
        elif kind[0] == "dead":
            # One huge hidden feature that no output reads.
            w.mlp_in[5] *= np.float32(2.0 ** kind[1])
            w.mlp_out[:, 5] = 0.0
        elif kind[0] == "picked":
            # One output that reads nothing but a tiny hidden feature.
            w.mlp_in[7] *= np.float32(2.0 ** -kind[1])
            w.mlp_out[:, 7] = 0.0
            w.mlp_out[9] = 0.0
            w.mlp_out[9, 7] = 2.0 ** kind[1]
        else:
            # One huge feature of the modulated norms that no GEMM reads.
            w.ada[[1, 4], 11] = 2.0 ** kind[1]
            w.qkv[:, 11] = w.mlp_gate[:, 11] = w.mlp_in[:, 11] = 0.0
    return (g, video, txt, emb, wv, wt), heads, hidden, mlp


@pytest.mark.parametrize("kind", [("features", 20), ("features", 40), ("features", -20), ("features", -40),
                                  ("dead", 36), ("picked", 20), ("picked", 40), ("norm", 24), ("norm", 40)])
def test_split_block_values_of_any_scale_in_a_row(gpu, kind):
    """Values far below their row's largest lose bits as fp16 planes, and
    vanish below 2^-40 of it. Where such values carry an output, it keeps the
    accuracy of fp32 products: the block's bound, per column."""
    print(f"case split block scales in a row {kind}", flush=True)
    args, heads, hidden, mlp = scaled_case(kind)
    got = run(*args, heads, hidden, mlp)
    ref = O.dit_block(*args, heads, HEAD_DIM, EPS, False)
    for a, b in zip(got, ref):
        err = np.max(np.abs(a.astype(np.float64) - b), 0) / np.max(np.abs(b), 0)
        print(f"  worst column {np.max(err):.3g}", flush=True)
        assert np.max(err) <= 1e-5


def test_split_block_infinity_times_a_tiny_value(gpu):
    """An infinite weight meets hidden values below 2^-40 of their row's
    largest: infinite outputs with the sign of the product, no NaN."""
    print("case split block inf times tiny", flush=True)
    (g, video, txt, emb, wv, wt), heads, hidden, mlp = scaled_case(("picked", 50))
    for w in (wv, wt):
        w.mlp_out[30, 7] = np.inf
    got = run(g, video, txt, emb, wv, wt, heads, hidden, mlp)
    with np.errstate(invalid="ignore"):
        ref = O.dit_block(g, video, txt, emb, wv, wt, heads, HEAD_DIM, EPS, False)
    for a, b in zip(got, ref):
        assert np.all(np.isinf(b[:, 30]))
        assert np.array_equal(a[:, 30].astype(np.float64), b[:, 30])
