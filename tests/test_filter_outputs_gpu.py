"""ls_filter_logits' dense outputs at aligned and unaligned row strides, with and
without the unfiltered rows (two ways to the same filtered rows), and nothing
written past a row's vocabulary."""

import pytest
import torch

from loopspec_amd import _lib, verify
from tests.conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab,dtype", [(8, torch.bfloat16), (2056, torch.float32), (10000, torch.float16)])
@pytest.mark.parametrize("pad", [0, 1, 4])
@pytest.mark.parametrize("top_p,top_k", [(0.6, 0), (0.98, 0), (1.0, 5), (1.0, 0)])
def test_filtered_rows_at_any_stride(gpu, vocab, dtype, pad, top_p, top_k):
    rows = 5
    g = torch.Generator().manual_seed(vocab + pad)
    x = (torch.randn(rows, vocab, generator=g) * 3).to(dtype).to(gpu)
    x[1, vocab // 2] = float("inf")
    x[2] = -float("inf")
    x[3, 1] = float("nan")
    announce(f"filter outputs V={vocab} {dtype} pad={pad} p={top_p} k={top_k}")
    both = verify.filter_logits(x, 1.0, top_p, top_k=top_k, want_probs=True)
    out = torch.full((rows + 1, vocab + pad), -3.0, device=gpu)
    ws = torch.zeros(_lib.query("ls_filter_logits_workspace", rows, vocab), dtype=torch.uint8, device=gpu)
    _lib.call("ls_filter_logits", x.data_ptr(), x.stride(0), _lib.dtype_code(x), rows, vocab, 1.0, top_p, None, top_k,
              None, 0, out.data_ptr(), out.stride(0), None, None, ws.data_ptr(), ws.numel(), _lib.stream(gpu))
    torch.cuda.synchronize()
    assert torch.equal(out[:rows, :vocab].view(torch.int32), both["filtered"].view(torch.int32))
    assert bool((out[:rows, vocab:] == -3.0).all()) and bool((out[rows] == -3.0).all())


@pytest.mark.parametrize("top_p", [0.6, 0.97])
def test_filtered_rows_over_their_logits(gpu, top_p):
    """The filtered rows written over float32 logits (the support re-read included)."""
    rows, vocab = 3, 20000
    x = (torch.randn(rows, vocab, generator=torch.Generator().manual_seed(1)) * 3).to(gpu)
    announce(f"filter in place p={top_p}")
    want = verify.filter_logits(x, 1.0, top_p)["filtered"]
    ws = torch.zeros(_lib.query("ls_filter_logits_workspace", rows, vocab), dtype=torch.uint8, device=gpu)
    _lib.call("ls_filter_logits", x.data_ptr(), x.stride(0), _lib.dtype_code(x), rows, vocab, 1.0, top_p, None, 0,
              None, 0, x.data_ptr(), x.stride(0), None, None, ws.data_ptr(), ws.numel(), _lib.stream(gpu))
    torch.cuda.synchronize()
    assert torch.equal(x.view(torch.int32), want.view(torch.int32))
