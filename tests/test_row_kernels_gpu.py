"""The kernels of a decode step that have a row or a few to work on, at the edges of what a thread and a workgroup take."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    from llm_infer_amd.kernels import ops
    return ops


# rows of whole quads and not, shared by one workgroup and by several, of a table that is 16-byte aligned and not
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,d,shift", [(1, 1, 0), (1, 7, 0), (3, 1024, 0), (2, 1028, 0), (5, 4100, 0), (255, 260, 0), (256, 260, 0), (300, 2049, 0),
                                       (2, 64, 4), (2, 66, 1)])
def test_gathered_rows(ops, dtype, n, d, shift):
    table = torch.randn(50 * d + shift, device=DEV, dtype=dtype)[shift:].view(50, d)
    ids = torch.randint(0, 50, (n,), device=DEV, dtype=torch.int32)
    assert torch.equal(ops.embed(table, ids), table[ids.long()].float())
    if d % 2:
        return
    pos = torch.randint(0, 5000, (n,), device=DEV, dtype=torch.int32)
    freq = 10000.0 ** (-torch.arange(0, d, 2, device=DEV, dtype=torch.float32) / d)
    got = ops.embed_positions(table, ids, pos, freq, 1.5).double()
    angle = pos.double()[:, None] * freq.double()
    want = table[ids.long()].double() * 1.5
    want[:, 0::2] += angle.sin()
    want[:, 1::2] += angle.cos()
    # the angle rounds to float32 once (half an ulp of it), sine, product and sum to some ulps of their size
    bound = angle.repeat_interleave(2, 1) * 2.0 ** -24 + 4 * 2.0 ** -23 * (1 + want.abs())
    assert ((got - want).abs() <= bound).all()


# one chunk, the edges between chunks and between a thread's elements, ties: the first of the largest
@pytest.mark.parametrize("v", [1, 63, 255, 257, 4095, 4096, 4097, 8193, 32000])
def test_argmax_first_of_the_largest(ops, v):
    x = torch.randint(0, 50, (5, v), device=DEV).float()
    x[1] = -torch.inf
    x[2, v // 2:] = 60.0
    x[3, -1] = 70.0
    x[4, 0] = 70.0
    assert ops.argmax(x).tolist() == [int((r == r.max()).nonzero()[0]) for r in x.cpu()]
