"""The dense path's softmax kernels where the blocks of a matrix are gathered on one XCD (rows that are not whole cache lines, large
matrices; whole groups of eight matrices and an incomplete one after them) and at the edges of the forward's numbers of keys
per thread, against float64."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,keys,queries", [(8, 33, 33), (9, 192, 65), (17, 193, 100), (7, 384, 97), (16, 385, 40), (11, 40, 512), (24, 768, 63), (8, 769, 34),
                                                (10, 64, 64), (9, 20, 32)])
@pytest.mark.parametrize("window,global_tokens", [(0, 0), (19, 2)])
def test_every_block_of_every_matrix(batch, keys, queries, window, global_tokens):
    from sentinel_amd import HipOps
    print(f"case {batch} {keys} {queries} {window} {global_tokens}", flush=True)
    gen = torch.Generator("cuda").manual_seed(batch * keys + queries)
    scores = 3 * torch.randn(batch, keys, queries, device="cuda", generator=gen)
    gradient = torch.randn(batch, keys, queries, device="cuda", generator=gen)
    scale = 0.25
    k, q = torch.arange(keys, device="cuda")[:, None], torch.arange(queries, device="cuda")[None, :]
    allowed = (k <= q) & ((k < global_tokens) | (k > q - window) | (window == 0))
    want = torch.softmax(torch.where(allowed, scores.double() * scale, -1.0e9), dim=1)
    HipOps.masked_softmax_in_place(scores, scale, window, global_tokens)
    # a probability is at most 1: a few roundings of the exponential, the sum and the product
    assert np.abs((scores - want).cpu().numpy()).max() <= 2e-6
    p = scores.double()
    want_ds = torch.where(allowed, p * (gradient - (gradient * p).sum(dim=1, keepdim=True)), 0.0) * scale
    HipOps.masked_softmax_backward_in_place(scores, gradient, scale, window, global_tokens)
    # |P| <= 1, |dP| <= 6, sums of up to 769 products rounded in fp32: far below 1e-5
    assert np.abs((gradient - want_ds).cpu().numpy()).max() <= 1e-5 * max(1.0, float(want_ds.abs().max()))
