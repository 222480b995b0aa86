"""The vocabulary head at the edges of its row rule: every tile height, row
counts on both sides of each, hidden sizes shorter than the load rings, and
column counts around a block."""

import pytest
import torch

from loopspec_amd import verify
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
