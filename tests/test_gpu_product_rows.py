"""Products whose rows are not whole vectors (product_rows_kernel in
pe_product.hip) and products with an operand that runs along another axis than
the output's inner one (product_tile_kernel): vectors that cross rows, short
rows, odd totals, partial tiles, unaligned bases and operand orders, bit-exact
against torch on the CPU."""
import ctypes

import pytest
import torch

from pto_einsum import abi, launch, runtime

pytestmark = pytest.mark.gpu

CASES = [
    # out shape, a strides, b strides
    ((1003,), (1,), (1,)),                                  # flat, odd total
    ((3,), (1,), (1,)),                                     # less than a vector
    ((7, 5), (5, 1), (0, 1)),                               # rows about a vector long
    ((50, 3), (3, 1), (0, 1)),                              # several rows in a vector
    ((40, 1), (1, 0), (1, 0)),
    ((9, 1153), (1153, 1), (0, 1)),                         # bsd,d
    ((9, 1153), (1153, 1), (1, 0)),                         # row scale
    ((9, 1153), (1, 0), (1153, 1)),                         # ... as the first operand
    ((33, 65), (1, 0), (0, 1)),                             # outer product
    ((32, 64), (1, 0), (0, 1)),                             # ... with whole vectors
    ((3, 20, 5, 33), (3300, 165, 33, 1), (0, 33, 0, 1)),    # bshd,sd
    ((3, 20, 5, 33), (0, 33, 0, 1), (3300, 165, 33, 1)),    # the other way round
    ((6, 40, 33), (33, 198, 1), (0, 33, 1)),                # A with permuted outer axes
    ((6, 40, 33), (33, 198, 1), (40, 1, 0)),                # ... times a scalar per row
    ((5, 30, 31), (930, 31, 1), (930, 31, 1)),              # merges into one axis
    ((70, 90), (90, 1), (1, 70)),                           # tiles: B transposed
    ((64, 64), (1, 64), (64, 1)),                           # A transposed
    ((130, 65), (1, 130), (1, 130)),                        # both: one axis order, two of them
    ((3, 70, 90), (6300, 90, 1), (1, 3, 210)),              # B contiguous along a short outer axis: one by one
    ((9, 70, 90), (6300, 90, 1), (1, 9, 630)),              # ... along the first axis
    ((5, 70, 4, 90), (25200, 360, 90, 1), (25200, 1, 6300, 70)),
    ((70, 90), (1, 0), (1, 70)),                            # A broadcast along the row
    ((70, 3000, 37), (111000, 37, 1), (0, 0, 1)),           # 30 000 blocks
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("add_zero", [0, 1])
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("shape,sa,sb", CASES)
def test_rows_bit_exact(shape, sa, sb, off, add_zero, dtype):
    g = torch.Generator().manual_seed(sum(shape) + add_zero)
    na = 1 + sum((n - 1) * s for n, s in zip(shape, sa))
    nb = 1 + sum((n - 1) * s for n, s in zip(shape, sb))
    a, b = torch.randn(na, generator=g).to(dtype), torch.randn(nb, generator=g).to(dtype)
    a[::7] = -0.0
    b[::11] = 2.0 ** -20 if dtype == torch.float16 else 2.0 ** -130
    n = 1
    for s in shape:
        n *= s
    code = launch.DT_F32 if dtype == torch.float32 else launch.DT_F16
    d = abi.product_desc(launch.ProductDesc(code, add_zero, list(shape), list(sa), list(sb), na, nb))
    # Operands at the requested offset, and a guard after the output.
    ga, gb = (torch.cat([x.new_zeros(off), x]).cuda()[off:] for x in (a, b))
    out = torch.full((n + 8,), float("nan"), device="cuda")
    rc = abi.bind().pe_product(ctypes.byref(d), *(ctypes.c_void_p(t.data_ptr()) for t in (ga, gb, out)),
                               ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, runtime.last_error()
    want = torch.as_strided(a, shape, sa).float() * torch.as_strided(b, shape, sb).float()
    if add_zero:
        want = 0.0 + want
    got = out.cpu()
    assert bool(torch.isnan(got[n:]).all())
    assert torch.equal(got[:n].view(torch.int32), want.contiguous().view(-1).view(torch.int32))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("nb,q,p", [(1000, 8, 8), (300, 12, 12), (300, 15, 17), (300, 16, 16), (40, 64, 8), (40, 8, 64)])
def test_many_small_transposed_matrices(nb, q, p, dtype):
    """bqp,bpq->bqp on both sides of the tile kernel's rule on full tiles."""
    test_rows_bit_exact((nb, q, p), (q * p, p, 1), (q * p, 1, q), 0, 0, dtype)
