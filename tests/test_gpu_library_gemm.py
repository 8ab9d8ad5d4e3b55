"""DiT blocks on either side of the rules that choose between the GEMMs of
csrc/dit_gemm.hip and the library's (fp32: 320 video rows, 384 at hidden 5120; bf16:
5000 video rows at hidden > 1536), and the library path in each form it takes: shifted, last
block, MLP weights stored apart and back to back. Against the oracle block
with the block tests' tolerances, fp32 1e-5 and bf16 2e-2 of the largest value."""

import ctypes

import numpy as np
import pytest

import awa_hip as A
import oracle as O
from awa_cases import geometry
from test_dit_block_oracle import EPS, HEAD_DIM
from test_gpu_dit_block import DeviceBranch, download_act, upload_act
from test_gpu_split_gemm import off, weights

pytestmark = pytest.mark.gpu

FP32 = dict(heads=2, hidden=512, mlp=1384)
WIDE = dict(heads=1, hidden=5120, mlp=64)
BF16 = dict(heads=1, hidden=1544, mlp=200)


def problem(grid, shifted, heads, hidden, mlp, seed=17):
    rng = np.random.default_rng(seed)
    g = geometry(grid + (2, 8, 8, 33), shifted)
    n = lambda *s: rng.standard_normal(s).astype(np.float32)
    return g, n(g.source_tokens, hidden), n(33, hidden), n(hidden * 6), weights(rng, heads, hidden, mlp), \
        weights(rng, heads, hidden, mlp)


def run(args, es, last, adjacent, heads, hidden, mlp):
    """One block object's outputs, and whether its GEMMs are the library's."""
    g, video, text, emb, wv, wt = args
    blk = A.DitBlock(*g.args, g.text_tokens, g.shifted, heads, HEAD_DIM, hidden, mlp, last,
                     A.COMPUTE_F32 if es == 4 else A.COMPUTE_BF16, EPS)
    dv, dt = DeviceBranch(wv, es, adjacent_mlp=adjacent), DeviceBranch(wt, es, adjacent_mlp=adjacent)
    on_library = A.lib().awa_dit_block_on_library(ctypes.c_void_p(blk.handle), ctypes.byref(dv.struct),
                                                  ctypes.byref(dt.struct))
    bv, bt, be = upload_act(video, es), upload_act(text, es), upload_act(emb, es)
    ov, ot = A.DeviceBuffer(video.size * es), A.DeviceBuffer(text.size * es)
    blk.forward(dv.struct, dt.struct, bv.ptr, bt.ptr, be.ptr, ov.ptr, ot.ptr)
    A.synchronize()
    out = download_act(ov, video.shape, es), download_act(ot, text.shape, es)
    blk.destroy()
    return out, bool(on_library)


@pytest.mark.parametrize("es,grid,shape,library", [
    (4, (1, 11, 29), FP32, True),                     # 319 rows
    (4, (1, 16, 20), FP32, False),                    # 320
    (4, (1, 1, 9), FP32, True),
    (4, (1, 19, 20), WIDE, True),                     # 380 rows, where the library is the faster
    (4, (2, 16, 12), WIDE, False),                    # 384
    (2, (5, 25, 40), BF16, False),                    # 5000
    (2, (6, 28, 30), BF16, True),                     # 5040
    (2, (6, 28, 30), dict(BF16, hidden=1536), False),
])
def test_each_side_of_the_rules(gpu, es, grid, shape, library):
    print(f"case block route es={es} {grid} {shape}", flush=True)
    args = problem(grid, False, **shape)
    got, on_library = run(args, es, False, True, **shape)
    assert on_library == library
    ref = O.dit_block(*args, shape["heads"], HEAD_DIM, EPS, False, bf16=es == 2)
    errs = [off(a, b) for a, b in zip(got, ref)]
    print(f"  rel err video {errs[0]:.3g} text {errs[1]:.3g}", flush=True)
    assert max(errs) <= (1e-5 if es == 4 else 2e-2)


@pytest.mark.parametrize("es,grid,shape", [(4, (1, 16, 16), FP32), (2, (6, 28, 30), BF16)])
@pytest.mark.parametrize("shifted,last,adjacent", [(True, False, False), (False, True, True), (True, True, False)])
def test_library_blocks(gpu, es, grid, shape, shifted, last, adjacent):
    """Shifted and last blocks; a second block object of the shape takes the
    first one's algorithms and gives its bits."""
    print(f"case library block es={es} shifted={shifted} last={last} adjacent={adjacent}", flush=True)
    args = problem(grid, shifted, **shape)
    got, on_library = run(args, es, last, adjacent, **shape)
    again, _ = run(args, es, last, adjacent, **shape)
    assert on_library
    assert all(np.array_equal(a, b) for a, b in zip(got, again))
    ref = O.dit_block(*args, shape["heads"], HEAD_DIM, EPS, last, bf16=es == 2)
    errs = [off(a, b) for a, b in zip(got, ref)]
    print(f"  rel err video {errs[0]:.3g} text {errs[1]:.3g}", flush=True)
    assert max(errs) <= (1e-5 if es == 4 else 2e-2)
