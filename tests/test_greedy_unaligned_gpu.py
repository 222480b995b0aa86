"""Greedy argmax and verify over rows at any element: first and last elements
around the 16-byte boundaries, rows shorter than a vector, several segments."""

import pytest
import torch

from loopspec_amd import verify
from tests.conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("vocab", [1, 3, 7, 9, 15, 17, 255, 2049, 4103, 50257])
@pytest.mark.parametrize("offset,pad", [(0, 0), (1, 0), (3, 1), (5, 2)])
def test_argmax_rows_any_alignment(gpu, dtype, vocab, offset, pad):
    rows = 23
    g = torch.Generator().manual_seed(vocab * 8 + offset)
    buf = torch.full((offset + rows * (vocab + pad) + 8,), 60000.0)  # larger than any logit, around the rows
    x = torch.randn(rows, vocab, generator=g)
    for r in range(rows):  # maxima at the ends, ties, NaN
        if r % 4 == 0:
            x[r, 0] = 9.0
        if r % 4 == 1:
            x[r, vocab - 1] = 9.0
        if r % 4 == 2:
            x[r, vocab // 2] = 9.0
            x[r, vocab - 1] = 9.0
        if r % 11 == 10:
            x[r, (5 * r) % vocab] = float("nan")
    buf.as_strided((rows, vocab), (vocab + pad, 1), offset).copy_(x)
    view = buf.to(dtype).to(gpu).as_strided((rows, vocab), (vocab + pad, 1), offset)
    announce(f"argmax any alignment {dtype} V={vocab} offset={offset} pad={pad}")
    got = verify.argmax_rows(view)
    torch.cuda.synchronize()
    assert torch.equal(got.cpu(), torch.argmax(x.to(dtype).float(), dim=-1))


@pytest.mark.parametrize("batch,k,vocab,dtype", [(1, 2, 50257, torch.float16), (96, 3, 32003, torch.bfloat16),
                                                 (300, 1, 1001, torch.float32), (2, 64, 9, torch.bfloat16)])
def test_greedy_verify_odd_vocabulary(gpu, batch, k, vocab, dtype):
    g = torch.Generator().manual_seed(batch)
    t = torch.randn(batch, k + 1, vocab, generator=g).to(dtype)
    d = torch.where(torch.rand(batch, k, 1, generator=g) < 0.7, t[:, :k], torch.randn(batch, k, vocab, generator=g).to(dtype))
    announce(f"greedy verify odd vocabulary B={batch} k={k} V={vocab} {dtype}")
    acc, tok = verify.greedy_verify(t.to(gpu), d.to(gpu))
    acc2, tok2 = verify.greedy_verify(t.to(gpu), None, d.float().argmax(-1).to(gpu))
    torch.cuda.synchronize()
    ids, did = t.float().argmax(-1), d.float().argmax(-1)
    want = (ids[:, :k] == did).long().cumprod(1).sum(1)
    toks = torch.where(torch.arange(k + 1) <= want[:, None], ids, -1)
    for a, b in ((acc, tok), (acc2, tok2)):
        assert torch.equal(a.cpu().long(), want) and torch.equal(b.cpu(), toks)
