"""Column layout with 16-bit arithmetic at the head dims around the line up to which 96 of a padded head's 128 dims are
computed on, at sequence lengths around the kernels' tiles; the kept 16-bit O is zero in the dims that were not."""
import numpy as np
import pytest
import torch

import gpu_util

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("head_dim", [72, 88, 96, 104])
@pytest.mark.parametrize("shape", [(2, 2, 1, 1, True, 0, 0), (4, 2, 129, 2, True, 0, 0), (2, 1, 193, 2, False, 0, 0),
                                   (2, 2, 260, 1, True, 70, 3)])
@pytest.mark.parametrize("compute", ["bf16", "fp16"])
def test_padded_head_dims(head_dim, shape, compute):
    import sentinel_amd
    from sentinel_amd import HipFlashAttention
    hq, hkv, t, packs, causal, window, global_tokens = shape
    d = head_dim
    print(f"case {compute} d{d} {shape}", flush=True)
    q, k, v, g = gpu_util.make_inputs(hq, hkv, d, t, packs, seed=d + t, dtype=compute)
    want = gpu_util.oracle(q, k, v, g, hq, hkv, d, t, packs, causal=causal, window=window, global_tokens=global_tokens)
    qd, kd, vd, gd = (torch.from_numpy(x).cuda() for x in (q, k, v, g))
    args = (hq, d, 1.0 / np.sqrt(np.float32(d)), causal, 0, t, packs)
    kw = dict(kv_head_count=hkv, compute=compute, window_size=window, global_token_count=global_tokens)
    code = {"bf16": 1, "fp16": 2}[compute]
    need = sentinel_amd.load_library().sentinel_hip_flash_workspace_bytes(0, code, 0, hq, hkv, d, t, packs, 1)
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device="cuda")  # (16-bit NaNs)
    out, lse = HipFlashAttention.forward_multi_head(qd, kd, vd, None, None, *args, workspace=ws, keep_for_backward=True, **kw)
    elements = packs * hq * t * 128
    kept = ws.view(torch.int16)[elements:2 * elements].view(-1, 128)
    assert (kept[:, d:] == 0).all()
    grads = HipFlashAttention.backward_multi_head(qd, kd, vd, out, lse, gd, None, None, None, None, *args, workspace=ws,
                                                  reuse_forward_workspace=True, **kw)
    torch.cuda.synchronize()
    for key, got in zip(("out", "dq", "dk", "dv"), (out, *grads)):
        gpu_util.assert_close_lowp(got.cpu().numpy(), want[key], key, d)
    gpu_util.assert_close_fp32(lse.cpu().numpy(), want["lse"], "lse", tol=1e-3)
