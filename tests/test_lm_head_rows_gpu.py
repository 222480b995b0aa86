"""The vocabulary head at the edges of its row rule: every tile height, row
counts on both sides of each, hidden sizes shorter than the load rings, and
column counts around a block."""

import pytest
import torch

from loopspec_amd import _lib, verify
from tests.conftest import announce
from tests.test_lm_head_gpu import check, make, reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden_size,vocab", [(64, 193), (128, 1000), (192, 384), (320, 577), (576, 2049)])
@pytest.mark.parametrize("rows", [1, 16, 17, 32, 33, 64, 65, 128, 129, 192, 193, 256, 257, 321, 641])
def test_lm_head_rows(gpu, rows, hidden_size, vocab):
    hidden, weight = make(rows, hidden_size, vocab, rows * 7 + vocab)
    announce(f"lm_head rows M={rows} H={hidden_size} V={vocab}")
    h, w = hidden.to(gpu), weight.to(gpu)
    ids = verify.lm_head_argmax(h, w)
    out = torch.full((rows + 1, vocab + 8), 7.0, device=gpu)
    f32 = verify.lm_head_logits(h, w, out=out[:rows, :vocab])
    torch.cuda.synchronize()
    logits, bound = reference(hidden, weight)
    check(ids.cpu().numpy(), logits, bound)
    err = (f32.double().cpu() - torch.from_numpy(logits)).abs()
    assert bool((err <= torch.as_tensor(bound)).all()), float((err - torch.as_tensor(bound)).max())
    assert torch.equal(f32.argmax(-1), ids)
    # nothing is written past the rows and columns asked for
    assert bool((out[rows] == 7.0).all()) and bool((out[:, vocab:] == 7.0).all())


@pytest.mark.parametrize("hidden_size", [192, 896, 1664])
@pytest.mark.parametrize("rows", [20, 33, 96, 128, 192, 256, 321])
def test_lm_head_bf16_logits_and_whole_ring_turns(gpu, rows, hidden_size):
    """bf16 logits of every tile height, at hidden sizes below, past and at twice
    the 12 k-blocks that the tallest unrolled loop takes per turn (3, 14, 26)."""
    vocab = 451
    hidden, weight = make(rows, hidden_size, vocab, rows + hidden_size)
    announce(f"lm_head bf16 logits M={rows} H={hidden_size} V={vocab}")
    h, w = hidden.to(gpu), weight.to(gpu)
    out = torch.full((rows + 1, vocab + 13), 7.0, dtype=torch.bfloat16, device=gpu)
    b16 = verify.lm_head_logits(h, w, out=out[:rows, :vocab])
    f32 = verify.lm_head_logits(h, w)
    ids = verify.lm_head_argmax(h, w)
    torch.cuda.synchronize()
    logits, bound = reference(hidden, weight)
    assert bool(((f32.double().cpu() - torch.from_numpy(logits)).abs() <= torch.as_tensor(bound)).all())
    assert torch.equal(b16, f32.to(torch.bfloat16))  # the same sums, rounded once
    assert torch.equal(f32.argmax(-1), ids)
    assert bool((out[rows] == 7.0).all()) and bool((out[:, vocab:] == 7.0).all())


def test_lm_head_more_workgroups_than_one_launch_dimension(gpu):
    """10,485,800 rows at 256 column blocks: 2^23 workgroups of 512 lanes and more
    than 2^32 lanes. The rows repeat 97 others, whose period meets every place of a
    row block, so the ids must repeat theirs."""
    period, rows, hidden_size, vocab = 97, 10_485_800, 64, 49152
    hidden, weight = make(period, hidden_size, vocab, 5)
    announce(f"lm_head M={rows} H={hidden_size} V={vocab}")
    h, w = hidden.to(gpu), weight.to(gpu)
    want = verify.lm_head_argmax(h, w)
    check(want.cpu().numpy(), *reference(hidden, weight))
    many = h.repeat(-(-rows // period), 1)[:rows]
    out = torch.empty(rows, dtype=torch.int64, device=gpu)
    ws = torch.empty(_lib.query("ls_lm_head_argmax_workspace", rows, vocab), dtype=torch.uint8, device=gpu)
    _lib.call("ls_lm_head_argmax", many.data_ptr(), many.stride(0), w.data_ptr(), w.stride(0), _lib.dtype_code(many),
              rows, hidden_size, vocab, out.data_ptr(), ws.data_ptr(), ws.numel(), _lib.stream(gpu))
    torch.cuda.synchronize()
    assert torch.equal(out, want.repeat(-(-rows // period))[:rows])
    del ws
    torch.cuda.empty_cache()
