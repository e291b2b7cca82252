"""The dense path's softmax kernels at the edges of their shapes (64, 128, 256, 512 and 1024 keys held in registers, more in
passes), against float64.  The backward is given probabilities that are not zero on forbidden pairs too: its sum runs over all keys."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("keys", [1, 2, 63, 64, 65, 128, 129, 255, 256, 257, 512, 513, 1000, 1024, 1025])
@pytest.mark.parametrize("queries,start,window,global_tokens,segment", [(33, 0, 0, 0, 0), (65, 40, 24, 3, 0), (97, 0, 0, 0, 32), (70, 0, 9, 2, 35)])
def test_softmax_and_backward_match_float64(keys, queries, start, window, global_tokens, segment):
    from sentinel_amd import HipOps
    print(f"case {keys} {queries} {start} {window} {global_tokens} {segment}", flush=True)
    rng = np.random.default_rng(keys * 7 + queries)
    batch, scale = 3, 0.25
    k, q = np.arange(keys)[:, None], np.arange(queries)[None, :]
    same = (k // segment == q // segment) if segment else np.ones((keys, queries), bool)
    kp, qp = (k % segment, q % segment) if segment else (k, q + start)
    allowed = same & (kp <= qp) & ((kp < global_tokens) | (window <= 0) | (kp > qp - window))
    scores = (3 * rng.standard_normal((batch, keys, queries))).astype(np.float32)
    gradient = rng.standard_normal((batch, keys, queries)).astype(np.float32)
    masked = np.where(allowed, scores.astype(np.float64) * scale, -1.0e9)
    e = np.exp(masked - masked.max(axis=1, keepdims=True))
    want = e / e.sum(axis=1, keepdims=True)
    got = torch.from_numpy(scores).cuda()
    args = (scale, window, global_tokens, start, segment)
    HipOps.masked_softmax_in_place(got, *args)
    torch.cuda.synchronize()
    # a probability is at most 1: a few roundings of the exponential, the sum and the product
    assert np.abs(got.cpu().numpy() - want).max() <= 2e-6

    for p in (got.cpu().numpy(), rng.random((batch, keys, queries)).astype(np.float32) / keys):
        dot = (gradient.astype(np.float64) * p).sum(axis=1, keepdims=True)
        want_ds = np.where(allowed, p * (gradient - dot), 0.0) * scale
        gd = torch.from_numpy(gradient).cuda()
        HipOps.masked_softmax_backward_in_place(torch.from_numpy(p).cuda(), gd, *args)
        torch.cuda.synchronize()
        got_ds = gd.cpu().numpy()
        # |P| <= 1, |dP| <= 6, sums of up to 1025 products rounded in fp32: far below 1e-5
        assert np.abs(got_ds - want_ds).max() <= 1e-5 * max(1.0, np.abs(want_ds).max())
        assert (got_ds[:, ~allowed] == 0).all()
