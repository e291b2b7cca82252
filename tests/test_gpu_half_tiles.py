"""64-row tiles (dK / dV: 64 keys; forward, dQ: 64 queries; two wavefronts per 32 rows, their results merged through LDS) next
to the 128-row tiles, against the oracle: lengths around the edges of both tiles, grouped heads (a tile walks the group's heads), more tiles than workgroups at
once, and windows whose global tokens end inside, at and past a tile."""
import numpy as np
import pytest
import torch

import gpu_util

pytestmark = pytest.mark.gpu

# (q_heads, kv_heads, head_dim, seq_len, packs, causal, window, global_tokens)
CASES = [(2, 1, d, t, 1, causal, 0, 0) for d in (64, 128) for t in (31, 63, 64, 65, 127, 129, 193) for causal in (True, False)]
CASES += [
    (32, 8, 128, 300, 8, True, 0, 0),    # 64-key tiles, more of them than compute units
    (16, 4, 64, 200, 40, True, 0, 0),    # the same at two workgroups per compute unit
    (16, 16, 128, 129, 16, True, 0, 0),  # 128-key tiles, the second with one key
    (16, 16, 64, 129, 32, True, 0, 0),
    (17, 17, 64, 2030, 1, True, 0, 0),   # forward, dQ: more tiles than compute units, sixteen per head
    (4, 1, 128, 450, 1, True, 70, 63),
    (4, 1, 128, 450, 1, True, 70, 64),
    (4, 1, 64, 450, 1, True, 33, 65),
    (4, 1, 64, 321, 2, True, 200, 130),
    (16, 16, 128, 260, 16, True, 40, 1),
]


@pytest.mark.parametrize("case", CASES)
def test_key_tiles(case):
    from sentinel_amd import flash_attention_backward, flash_attention_forward
    hq, hkv, d, t, packs, causal, window, global_tokens = case
    print(f"case {case}", flush=True)
    q, k, v, g = gpu_util.make_inputs(hq, hkv, d, t, packs, seed=sum(case), dtype="bf16")
    want = gpu_util.oracle(q, k, v, g, hq, hkv, d, t, packs, causal=causal, window=window, global_tokens=global_tokens)
    qd, kd, vd, gd = (gpu_util.columns_to_device_bhtd(x, h, d, t, packs, 0, "bf16") for x, h in ((q, hq), (k, hkv), (v, hkv), (g, hq)))
    kw = dict(causal=causal, window_size=window, global_token_count=global_tokens)
    out, lse = flash_attention_forward(qd, kd, vd, **kw)
    dq, dk, dv = (torch.full_like(x, float("nan")) for x in (qd, kd, vd))
    flash_attention_backward(qd, kd, vd, out, lse, gd, dq=dq, dk=dk, dv=dv, **kw)
    torch.cuda.synchronize()
    assert np.abs(gpu_util.bht_to_columns(lse, hq, q.shape[1], 0) - want["lse"]).max() <= 2e-3
    for name, got, like in (("out", out, q), ("dq", dq, q), ("dk", dk, k), ("dv", dv, v)):
        gpu_util.assert_close_lowp(gpu_util.bhtd_to_columns(got, like, 0), want[name], name, d)


@pytest.mark.parametrize("compute", ["bf16", "fp16"])
@pytest.mark.parametrize("d,t", [(64, 65), (64, 300), (80, 193), (128, 129), (128, 450)])
def test_forward_does_not_depend_on_the_tiles(d, t, compute):
    """A sequence alone (64-query tiles) and among enough copies of itself (128-query tiles): P is rounded against the same
    reference, so the results differ by the order of fp32 sums of t terms, t * 2^-24 of the largest |v| (or of the LSE)."""
    from sentinel_amd import HipFlashAttention
    heads, packs = 4, 150
    assert heads * ((t + 127) // 128) <= 256 < heads * packs * ((t + 127) // 128)
    q, k, v = (torch.from_numpy(x).cuda() for x in gpu_util.make_inputs(heads, heads, d, t, 1, seed=d + t, sigma_qk=2.0)[:3])
    scale = 1.0 / np.sqrt(d)
    alone, lse = HipFlashAttention.forward_multi_head(q, k, v, None, None, heads, d, scale, True, 0, t, 1, compute=compute)
    many = [x.repeat(1, packs) for x in (q, k, v)]
    among, lse_among = HipFlashAttention.forward_multi_head(*many, None, None, heads, d, scale, True, 0, t, packs, compute=compute)
    assert (alone - among[:, -t:]).abs().max() <= t * 2.0 ** -24 * v.abs().max()
    assert (lse - lse_among[:, -t:]).abs().max() <= t * 2.0 ** -24 * max(1.0, float(lse.abs().max()))


@pytest.mark.parametrize("packs", [1, 150])  # 64-query tiles, 128-query tiles
@pytest.mark.parametrize("d", [64, 128])
def test_scores_far_below_zero(d, packs):
    """Raw scores below -1e30 are scores like any other: all of a row's are equal here, so O is the running mean of V."""
    from sentinel_amd import flash_attention_forward
    heads, t = 4, 130
    q = torch.full((packs, heads, t, d), 2.0 ** 55, device="cuda", dtype=torch.bfloat16)
    v = torch.randn(packs, heads, t, d, device="cuda", generator=torch.Generator("cuda").manual_seed(1)).abs().to(torch.bfloat16)
    out, _ = flash_attention_forward(q, -q, v, scale=1e-30)
    want = v.float().cumsum(2) / torch.arange(1, t + 1, device="cuda")[:, None]
    # the scaled scores are about -1e5 in fp32, whose rounding leaves 2 % in each probability at most
    assert ((out.float() - want).abs() <= 2e-2 * want).all()
