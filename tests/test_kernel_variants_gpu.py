"""GPU parity of single kernel variants and dispatch branches, at the sizes where each can go wrong."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def af3():
    import af3_kernels_amd
    af3_kernels_amd._lib.load()
    return af3_kernels_amd


def f32np(t):
    return t.detach().float().cpu().numpy()


@pytest.mark.parametrize("H,L,D,pad,first", [
    (1, 1, 24, 0, 0), (2, 2, 24, 1, 1), (3, 31, 32, 0, 1), (2, 33, 8, 3, 0), (1, 63, 24, 0, 0), (1, 65, 48, 0, 1),   # one wavefront, last tile nearly empty
    (2, 129, 24, 0, 0), (2, 190, 32, 5, 1), (3, 257, 24, 0, 0),   # key tiles split over four wavefronts
    (2, 129, 48, 0, 1), (2, 322, 64, 0, 0),                       # a pair of wavefronts per workgroup
    (16, 513, 48, 1, 0),                                          # two pairs, head_dim padded to 64
    (16, 515, 24, 1, 1),                                          # pairs on shared tiles, four computing wavefronts
    (16, 1027, 24, 0, 0), (16, 1024, 24, 7, 1),                   # ... eight
    (16, 1027, 48, 0, 1),                                         # loading wavefronts, one query block each
    (16, 2051, 24, 0, 0), (16, 2050, 48, 1, 0),                   # four wavefronts that load for themselves
])
def test_single_row_bias_at_any_address(af3, oracle, H, L, D, pad, first):
    """One batch row, bias rows that start at any element: what surrounds the L x L corner (here NaN) must not be used."""
    g = torch.Generator().manual_seed(L + D)
    q, k, v = (torch.randn(1, H, L, D, generator=g).to(torch.bfloat16) for _ in range(3))
    M = L + pad
    flat = torch.full((first + H * M * M,), float("nan")).to(torch.bfloat16)
    bias = flat[first:].view(H, M, M)
    bias[:, :L, :L] = torch.randn(H, L, L, generator=g).to(torch.bfloat16)
    keep = torch.rand(L, generator=g) < 0.8
    keep[L // 2] = True
    dev = flat.cuda()[first:].view(H, M, M)
    print("case", H, L, D, pad, first, flush=True)
    out = af3.dot_product_attention_cpp(q.cuda(), k.cuda(), v.cuda(), keep.cuda(), dev)
    torch.cuda.synchronize()
    want = oracle.dpa_formula(f32np(q), f32np(k), f32np(v), keep.numpy(), f32np(bias[:, :L, :L]))
    assert np.abs(f32np(out) - want).max() <= 2e-2
