"""The fp32 kernels' tilings (16, 32 or 64 own tokens per workgroup, tiles of 32 tokens in 16-byte pieces, single words or
through registers) at the sizes where each can go wrong, against the oracle at the fp32 bar of 1e-4.  Columns outside the
pack window hold NaN: a tile that reads past its sequence shows up in every result it touches."""
import numpy as np
import pytest
import torch

import gpu_util

pytestmark = pytest.mark.gpu

CASES = [
    # q heads, kv heads, d, T, packs, column start, spare columns, window, global tokens
    (1, 1, 1, 1, 1, 0, 0, 0, 0),
    (2, 2, 16, 15, 3, 1, 2, 0, 0),       # one partial tile, words
    (2, 1, 8, 16, 2, 4, 4, 0, 0),        # pieces, padded head dims
    (2, 2, 20, 33, 1, 0, 3, 0, 0),       # one token in the second tile
    (3, 3, 32, 64, 1, 0, 0, 0, 0),
    (4, 2, 40, 65, 2, 3, 1, 0, 0),
    (6, 2, 48, 100, 1, 8, 4, 30, 5),     # grouped heads, window edges inside tiles
    (2, 2, 64, 129, 1, 1, 0, 32, 0),
    (4, 1, 64, 96, 2, 0, 4, 17, 33),     # global tokens past a tile edge
    (2, 2, 72, 47, 1, 0, 0, 0, 0),
    (2, 1, 96, 80, 1, 4, 0, 0, 0),
    (2, 2, 128, 68, 1, 0, 4, 40, 1),
    (1, 1, 120, 35, 1, 2, 1, 0, 0),
    # grids large enough for the 32-token blocks and for the unsplit ones
    (8, 8, 16, 33, 100, 0, 0, 0, 0),
    (8, 4, 16, 65, 110, 1, 0, 0, 0),
    (8, 8, 32, 36, 60, 0, 4, 0, 0),
    (8, 8, 64, 65, 40, 0, 0, 20, 2),
    (8, 4, 64, 68, 40, 4, 0, 0, 0),
    (8, 8, 128, 40, 30, 0, 0, 0, 0),
]


# (the sliding window refines the causal mask)
@pytest.mark.parametrize("case,causal", [(c, causal) for c in CASES for causal in (True, False) if causal or not c[7]])
def test_columns_match_oracle(case, causal):
    from sentinel_amd import HipFlashAttention
    hq, hkv, d, t, packs, col0, pad, window, global_tokens = case
    print(f"case {case} causal={causal}", flush=True)
    q, k, v, g = gpu_util.make_inputs(hq, hkv, d, t, packs, seed=sum(case), col0=col0, pad=pad)
    want = gpu_util.oracle(q, k, v, g, hq, hkv, d, t, packs, col0=col0, causal=causal, window=window, global_tokens=global_tokens)
    for x in (q, k, v, g):
        x[:, :col0] = np.nan
        x[:, col0 + packs * t:] = np.nan
    qd, kd, vd, gd = (torch.from_numpy(x).cuda() for x in (q, k, v, g))
    out, dq, dk, dv = (torch.full_like(x, np.nan) for x in (qd, qd, kd, vd))
    lse = torch.full((hq, q.shape[1]), np.nan, device="cuda")
    geometry = (hq, d, 1.0 / np.sqrt(np.float32(d)), causal, col0, t, packs)
    kw = dict(kv_head_count=hkv, window_size=window, global_token_count=global_tokens)
    HipFlashAttention.forward_multi_head(qd, kd, vd, out, lse, *geometry, **kw)
    HipFlashAttention.backward_multi_head(qd, kd, vd, out, lse, gd, dq, dk, dv, None, *geometry, **kw)
    torch.cuda.synchronize()
    for key, got in (("out", out), ("lse", lse), ("dq", dq), ("dk", dk), ("dv", dv)):
        got = got.cpu().numpy()
        assert np.isnan(got[:, :col0]).all() and np.isnan(got[:, col0 + packs * t:]).all(), f"{key}: wrote outside the window"
        gpu_util.assert_close_fp32(got, want[key], key)


@pytest.mark.parametrize("batch,hq,hkv,t,causal", [(1, 2, 2, 65, True), (2, 4, 2, 65, False), (3, 2, 1, 1, True), (1, 1, 1, 32, True)])
def test_one_head_dim_in_the_native_layout(batch, hq, hkv, t, causal):
    """[B, H, T, 1]: tokens and head dims both have stride 1, as in no other call of either layout."""
    from sentinel_amd import flash_attention_backward, flash_attention_forward
    print(f"case {batch} {hq} {hkv} {t} causal={causal}", flush=True)
    q, k, v, g = gpu_util.make_inputs(hq, hkv, 1, t, batch, seed=t + batch)
    want = gpu_util.oracle(q, k, v, g, hq, hkv, 1, t, batch, causal=causal)
    qd, kd, vd, gd = (gpu_util.columns_to_device_bhtd(x, h, 1, t, batch, 0, "fp32") for x, h in ((q, hq), (k, hkv), (v, hkv), (g, hq)))
    out, lse = flash_attention_forward(qd, kd, vd, causal=causal)
    dq, dk, dv = flash_attention_backward(qd, kd, vd, out, lse, gd, causal=causal)
    torch.cuda.synchronize()
    gpu_util.assert_close_fp32(gpu_util.bht_to_columns(lse, hq, q.shape[1], 0), want["lse"], "lse")
    for key, got, like in (("out", out, q), ("dq", dq, q), ("dk", dk, k), ("dv", dv, v)):
        gpu_util.assert_close_fp32(gpu_util.bhtd_to_columns(got, like, 0), want[key], key)
