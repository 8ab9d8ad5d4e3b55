"""Layers of long mixed windows, which run the 8-wave attention kernels in
spite of idle waves: the last query block of a window ends inside a wave, and
windows shorter than one block sit beside long ones. Against the float64
definition of the layer with the gates of the fused layers (fp32 1e-4 max abs;
bf16 2e-2 of the largest value)."""

import numpy as np
import pytest

import awa_hip as A
from awa_cases import geometry, qkv_inputs
from device_blobs import mat3, qkv_blob, read_mat3, read_video, video_out_blob
from float64_model import layer64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("compute", [A.COMPUTE_F32, A.COMPUTE_BF16])
@pytest.mark.parametrize("grid", [(12, 29, 19, 2, 4, 4, 58), (3, 46, 48, 2, 2, 2, 58)])
def test_long_mixed_windows_match_float64(gpu, compute, grid):
    shifted, heads, checked = True, 20, [0, 19]
    print(f"case long windows {grid} compute={compute}", flush=True)
    g = geometry(grid, shifted)
    es = 4 if compute == A.COMPUTE_F32 else 2
    video, text = qkv_inputs(g, heads, 128, 11)
    if es == 2:
        video, text = (A.bf16_bits_to_f32(A.f32_to_bf16_bits(x)).reshape(x.shape) for x in (video, text))
    plan = A.Plan(A.LayerParams(*g.args, g.text_tokens, g.shifted), heads=heads)
    plan.upload()
    vq, tq = qkv_blob(video, "a", es), qkv_blob(text, "a", es)
    vo = video_out_blob(g.t, g.h, g.w, heads, 128, es, False)
    to = mat3(128, heads, g.text_tokens, es)
    plan.forward(vq.blob, tq.blob, vo.blob, to.blob, compute)
    A.synchronize()
    got = read_video(vo, g.t, g.h, g.w, heads, 128), read_mat3(to)
    ref = layer64(g, video[:, :, checked], text[:, :, checked])
    for a, b in zip(got, ref):
        err = np.max(np.abs(a.reshape(-1, heads, 128)[:, checked] - b))
        print(f"  max abs err {err:.3g}", flush=True)
        assert err <= (1e-4 if es == 4 else 2e-2 * np.max(np.abs(b)))
