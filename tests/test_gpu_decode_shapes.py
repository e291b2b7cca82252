"""Cache attention where its workgroups change shape or end: context lengths around one pass of 64 positions, one or more teams of
wavefronts in a workgroup, split chunks of 64 and of 256 positions; head dims that are no multiple of 16; odd row strides.  Against
float64; positions past the used prefix hold NaN."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(4, 4, 8), (4, 2, 24), (6, 6, 64), (8, 2, 72), (8, 1, 80), (4, 4, 128), (16, 2, 128), (3, 3, 32)]
LENGTHS = [1, 3, 63, 64, 65, 127, 128, 129, 256, 257, 700, 8192, 8193, 8400, 8705]


@pytest.mark.parametrize("hq,hkv,d", SHAPES)
@pytest.mark.parametrize("length", LENGTHS)
def test_decode_matches_float64(hq, hkv, d, length):
    from sentinel_amd import decode_attention
    for spare, window, global_tokens in ((0, 0, 0), (3, 0, 0), (64, max(1, length // 3), 5), (1, 70, 0)):
        print(f"case {hq} {hkv} {d} {length} spare={spare} window={window} global={global_tokens}", flush=True)
        rng = np.random.default_rng(length * 31 + d + spare)
        capacity = length + spare
        q = rng.standard_normal((hq * d, 1)).astype(np.float32)
        k, v = (rng.standard_normal((hkv * d, capacity)).astype(np.float32) for _ in range(2))
        for x in (k, v):
            x[:, length:] = np.nan
        visible = np.ones(length, bool)
        if 0 < window < length:
            position = np.arange(length)
            visible = (position < global_tokens) | (position >= length - window)
        kd = k[:, :length].astype(np.float64).reshape(hkv, d, length)
        vd = v[:, :length].astype(np.float64).reshape(hkv, d, length)
        want = np.empty((hq, d))
        for h in range(hq):
            s = np.where(visible, q.reshape(hq, d)[h].astype(np.float64) @ kd[h * hkv // hq] / np.sqrt(d), -np.inf)
            p = np.exp(s - s.max())
            want[h] = vd[h * hkv // hq] @ (p / p.sum())
        got = decode_attention(torch.from_numpy(q).cuda(), torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda(), length, hq, d,
                               kv_head_count=hkv, window_size=window, global_token_count=global_tokens)
        torch.cuda.synchronize()
        # averages of values of order one, sums of up to 8705 terms in fp32: well below the 1e-4 of the fp32 path
        assert np.abs(got.cpu().numpy().reshape(hq, d) - want).max() <= 2e-5


def _attend64(q, k, v, length, visible, d):
    """softmax(q K / sqrt(d)) V of the visible positions, single head, float64"""
    s = np.where(visible, q[:, 0].astype(np.float64) @ np.where(visible, k[:, :length], 0.0) / np.sqrt(d), -np.inf)
    p = np.exp(s - s.max())
    return np.where(visible, v[:, :length], 0.0).astype(np.float64) @ (p / p.sum())


@pytest.mark.parametrize("d", [8, 24, 40, 72, 104, 120, 64])
@pytest.mark.parametrize("length", [50, 200, 9000])
def test_a_key_of_minus_infinity_hides_its_position(d, length):
    """In the last rows of K, which share a matrix instruction with head dims past the last."""
    from sentinel_amd import decode_attention
    print(f"case {d} {length}", flush=True)
    rng = np.random.default_rng(d + length)
    q = np.abs(rng.standard_normal((d, 1))).astype(np.float32)
    k, v = (rng.standard_normal((d, length)).astype(np.float32) for _ in range(2))
    hidden = [0, 5, length // 2, length - 1]
    for i, position in enumerate(hidden):
        k[d - 1 - i, position] = -np.inf
    visible = np.ones(length, bool)
    visible[hidden] = False
    want = _attend64(q, np.where(np.isinf(k), 0, k), v, length, visible, d)
    got = decode_attention(torch.from_numpy(q).cuda(), torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda(), length, 1, d)
    assert np.abs(got.cpu().numpy()[:, 0] - want).max() <= 2e-5


@pytest.mark.parametrize("hq,hkv,d,length,window,global_tokens", [
    (4, 4, 64, 200, 30, 0),        # one workgroup for the whole context
    (4, 4, 16, 256, 70, 66),
    (2, 2, 128, 1000, 100, 20),    # chunks of 64
    (4, 2, 64, 9000, 300, 300),    # chunks of 256
])
def test_hidden_positions_do_not_count(hq, hkv, d, length, window, global_tokens):
    """Infinities and NaN in the cache at positions the sparse mask hides."""
    from sentinel_amd import decode_attention
    print(f"case {hq} {hkv} {d} {length} {window} {global_tokens}", flush=True)
    rng = np.random.default_rng(d + length)
    position = np.arange(length)
    visible = (position < global_tokens) | (position >= length - window)
    q = rng.standard_normal((hq * d, 1)).astype(np.float32)
    k, v = (rng.standard_normal((hkv * d, length)).astype(np.float32) for _ in range(2))
    hidden = np.flatnonzero(~visible)
    for x in (k, v):
        x[::3, hidden[::5]] = np.inf
        x[1::3, hidden[::7]] = np.nan
        x[:, [hidden[0], hidden[-1]]] = -np.inf
    got = decode_attention(torch.from_numpy(q).cuda(), torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda(), length, hq, d,
                           kv_head_count=hkv, window_size=window, global_token_count=global_tokens).cpu().numpy().reshape(hq, d)
    for h in range(hq):
        head = slice(h * hkv // hq * d, (h * hkv // hq + 1) * d)
        assert np.abs(got[h] - _attend64(q[h * d:(h + 1) * d], k[head], v[head], length, visible, d)).max() <= 2e-5


@pytest.mark.parametrize("hq,hkv,d", [(12, 12, 64), (4, 4, 16), (16, 2, 128), (16, 4, 64), (12, 6, 80)])
def test_long_sums_keep_their_precision(hq, hkv, d):
    """Sums over thousands of positions in short chains: about four roundings (4 * 2^-24) in the 2-norm, where one chain per workgroup and
    a rounded factor at every change of the reference leave five."""
    from sentinel_amd import decode_attention
    length = 9001
    squared = 0.0
    seeds = 8
    for seed in range(seeds):
        gen = torch.Generator("cuda").manual_seed(seed)
        q = torch.randn(hq * d, 1, device="cuda", generator=gen)
        k, v = (torch.randn(hkv * d, length, device="cuda", generator=gen) for _ in range(2))
        kd, vd = (x.double().reshape(hkv, d, length).repeat_interleave(hq // hkv, 0) for x in (k, v))
        scale = float(np.float32(1.0 / np.sqrt(d)))
        p = torch.softmax((q.double().reshape(hq, 1, d) @ kd).squeeze(1) * scale, 1)
        want = (vd @ p.unsqueeze(2)).reshape(hq * d, 1)
        got = decode_attention(q, k, v, length, hq, d, kv_head_count=hkv, scale=scale)
        squared += float(((got.double() - want).norm() / want.norm()) ** 2)
    assert (squared / seeds) ** 0.5 <= 4 * 2.0 ** -24
