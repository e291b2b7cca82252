"""sentinel_hip_rope_rotate where its workgroups end inside a group of pairs, a column block or a run of heads.  The rotation
is two products and one sum per value in fp32, so torch's separate operations give the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,head_dim,columns,segment", [(1, 2, 1, 0), (3, 10, 63, 0), (2, 24, 65, 13), (12, 64, 130, 65),
                                                            (5, 40, 2050, 1025), (24, 64, 4100, 0), (3, 126, 700, 100)])
@pytest.mark.parametrize("inverse", [False, True])
def test_rotation_matches_separate_operations(heads, head_dim, columns, segment, inverse):
    from sentinel_amd import HipOps
    print(f"case {heads} {head_dim} {columns} {segment} {inverse}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(heads * 7 + columns)
    offset = 0 if segment else 3
    positions = segment if segment else columns + offset
    pairs = head_dim // 2
    angle = 10 * torch.rand(positions, pairs, device="cuda", generator=gen)
    cos, sin = torch.cos(angle).contiguous(), torch.sin(angle).contiguous()
    x = torch.randn(heads * head_dim, columns, device="cuda", generator=gen)
    at = torch.arange(columns, device="cuda") % segment if segment else torch.arange(columns, device="cuda") + offset
    c, s = cos[at].t()[None], sin[at].t()[None]
    even, odd = x.view(heads, pairs, 2, columns)[:, :, 0], x.view(heads, pairs, 2, columns)[:, :, 1]
    if inverse:
        want = torch.stack((even * c + odd * s, -even * s + odd * c), dim=2)
    else:
        want = torch.stack((even * c - odd * s, even * s + odd * c), dim=2)
    want = want.reshape(heads * head_dim, columns)
    HipOps.rotary_rotate_in_place(x, heads, head_dim, pairs, cos, sin, 0 if segment else offset, segment, inverse=inverse)
    torch.cuda.synchronize()
    assert torch.equal(x, want)
