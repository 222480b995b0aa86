"""GPU parity of rows whose support lies beyond their candidates: re-read
chunks, the two-pass whole-row select, the digit rounds behind it, top-k
resolved before top-p, and draws over the whole row. All against the oracle,
bit for bit."""

import numpy as np
import pytest
import torch

from oracle import numerics as nm
from oracle import sampling as osmp
from loopspec_amd import philox, verify, workloads
from tests import candidates
from tests.conftest import announce
from tests.test_sweep_gpu import epv_of, histories, oracle_drafts

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize("batch,k,vocab,dtype,t,top_p,top_k,penalty", [
    (2, 2, 49152, F32, 1.0, 0.9, 0, 1.0),      # about 2048 in the support: either side of the LDS list
    (2, 1, 49152, F32, 1.0, 0.95, 0, 1.0),     # dense supports of both rows
    (1, 4, 32000, BF16, 0.8, 0.95, 0, 1.0),    # chunks re-read
    (1, 2, 130000, BF16, 1.0, 0.95, 0, 1.0),   # a partial last chunk, 64 chunks
    (1, 1, 262144, F16, 1.0, 0.98, 0, 1.0),    # the largest vocabulary
    (3, 2, 2056, F32, 1.0, 0.999, 0, 1.0),     # a second chunk of one or two vectors
    (2, 2, 20000, BF16, 1.0, 0.95, 0, 1.3),    # penalised rows, dense
    (2, 2, 20000, F32, 1.0, 1.0, 0, 0.8),      # unfiltered rows with a penalty below 1
    (130, 1, 8192, F32, 1.0, 0.97, 0, 1.0),    # more units than CUs (two workgroups per CU)
    (1, 4, 32000, BF16, 0.8, 0.95, 50, 1.0),   # top-k decides inside the candidates
    (2, 1, 32000, F32, 1.0, 0.99, 3000, 1.0),  # top-k beyond the candidates, both whole-row selects
    (2, 1, 49152, F32, 1.0, 0.2, 2500, 1.0),   # top-p inside the candidates, top-k beyond them
    (130, 1, 8192, BF16, 1.0, 0.97, 600, 1.1),
    (130, 1, 8192, F32, 1.0, 1.0, 0, 1.0),     # unfiltered rows, two workgroups per CU
    (130, 1, 2056, BF16, 1.0, 1.0, 0, 1.2),
])
def test_spec_verify_large_supports(gpu, batch, k, vocab, dtype, t, top_p, top_k, penalty):
    pen = penalty != 1.0
    cfg = workloads.SamplingConfig("large-support", batch, k, vocab, dtype, t, top_p, penalty=penalty, top_k=top_k,
                                   hist_min=10 if pen else 0, hist_max=400 if pen else 0)
    inp = workloads.sampling_inputs(cfg, vocab + top_k)
    hists = histories(cfg, inp)
    drafts = oracle_drafts(cfg, inp, hists)
    inp["uniforms"][: (batch + 1) // 2, 0] = 0.9999999  # rejections: residual draws
    announce(f"large support B={batch} k={k} V={vocab} {dtype} T={t} p={top_p} k={top_k} pen={penalty}")
    acc, tok = verify.speculative_verify(
        inp["target"].to(gpu), inp["draft"].to(gpu), drafts.to(gpu), inp["uniforms"].to(gpu), t, top_p,
        penalty=penalty, history=inp["history"].to(gpu) if pen else None,
        history_len=inp["history_len"].to(gpu) if pen else None, top_k=top_k)
    torch.cuda.synchronize()
    want = osmp.speculative_verify(inp["target"].float().numpy(), inp["draft"].float().numpy(), drafts.numpy(),
                                   inp["uniforms"].numpy(), t, top_p, penalty, hists, top_k=top_k, epv=epv_of(dtype))
    assert np.array_equal(acc.cpu().numpy(), want.accept_len)
    assert np.array_equal(tok.cpu().numpy(), want.tokens)


def _rows(kind, v, rng):
    x = (rng.standard_normal(v) * 3).astype(np.float32)
    if kind == "plateau":      # thousands of equal logits at the cutoff: the digit rounds, all three
        x[:] = np.where(np.arange(v) % 5 == 0, np.float32(2.0), np.float32(-20.0))
    elif kind == "ladder":     # a plateau of near-equal distinct logits: more in the window than the list holds
        x[:] = 1.0 + np.arange(v, dtype=np.float32) * np.float32(1e-7)
    elif kind == "nan_inf":    # no mass; -inf has none
        x[::7] = np.nan
        x[3::11] = -np.inf
    elif kind == "wide":       # p below 2^-63 and zero p
        x *= 40.0
    return x


@pytest.mark.parametrize("kind", ["plateau", "ladder", "nan_inf", "wide"])
@pytest.mark.parametrize("top_p,top_k", [(0.97, 0), (1.0 - 2.0 ** -24, 0), (0.97, 5000)])
def test_filter_and_sample_large_support_edges(gpu, kind, top_p, top_k):
    v = 16392
    rng = np.random.default_rng(5)
    x = torch.from_numpy(np.stack([_rows(kind, v, rng) for _ in range(2)]))
    u = torch.from_numpy(philox.uniforms((2,), seed=3))
    announce(f"large support edges {kind} p={top_p} k={top_k}")
    res = verify.filter_logits(x.to(gpu), 1.0, top_p, top_k=top_k)
    got = verify.sample_logits(x.to(gpu), u.to(gpu), 1.0, top_p, top_k=top_k)
    torch.cuda.synchronize()
    for r in range(2):
        want = osmp.filter_row(osmp.process_logits(x[r].numpy(), 1.0, epv=4), top_p, top_k)
        assert np.array_equal(res["filtered"][r].cpu().numpy(), want.P), r
        assert res["cutoff"][r].item() == want.cutoff, r
        assert res["mass"][r].item() == nm.mass_to_f32(want.mass_fx), r
        assert got[r].item() == osmp.categorical_pick(want.P, u[r].item()), r


@pytest.mark.parametrize("ulps", [256, 512])
@pytest.mark.parametrize("ties", [1500, 3000])  # inside the list's 2048, and past it
def test_top_k_at_a_subnormal_plateau(gpu, ulps, ties):
    """The k-th largest p is a plateau at 256 or 512 * 2^-149, the first value of a
    digit, whose logits' powers of two lie half of 2^-149 below it."""
    v = 16392
    x = np.full((2, v), -1000.0, dtype=np.float32)
    x[:, 0] = 0.0
    x[:, 3:3 + 5 * ties:5] = np.float32(np.log((ulps - 0.4) * 2.0 ** -149))
    announce(f"subnormal plateau ulps={ulps} ties={ties}")
    res = verify.filter_logits(torch.from_numpy(x).to(gpu), 1.0, 1.0, top_k=1000)
    torch.cuda.synchronize()
    want = osmp.filter_row(osmp.process_logits(x[0], 1.0, epv=4), 1.0, 1000)
    assert want.cutoff == np.float32(ulps * 2.0 ** -149)
    for r in range(2):
        assert res["cutoff"][r].item() == want.cutoff, r
        assert np.array_equal(res["filtered"][r].cpu().numpy(), want.P), r
        assert res["mass"][r].item() == nm.mass_to_f32(want.mass_fx), r


@pytest.mark.parametrize("rows", [2, 300])  # one finaliser workgroup per CU, and two
@pytest.mark.parametrize("dtype,penalty", [(F32, 1.0), (BF16, 1.0), (F32, 1.3)])
@pytest.mark.parametrize("top_k", [0, 40, 50, 51, 150, 151, 700])  # 50 tokens at 6.0, then 100 ties at 5.0
def test_re_read_chunks_with_top_k(gpu, rows, dtype, penalty, top_k):
    """Rows with a chunk that keeps no candidates: it is re-read, and the k-th
    largest is known only from the re-read list (above, at and below the top-p cutoff)."""
    row, top_p = candidates.path_rows()["refill"]
    x = torch.from_numpy(row).to(dtype)
    assert candidates.row_path(x.float().numpy(), top_p, epv=epv_of(dtype)) == "refill"
    hist = np.flatnonzero(row == 6.0)[::3].astype(np.int32)
    batch = torch.stack([x, x.flip(0)]).repeat(rows // 2, 1)
    hists = [hist, (len(row) - 1 - hist).astype(np.int32)]
    u = torch.from_numpy(philox.uniforms((rows,), seed=top_k))
    announce(f"re-read rows={rows} {dtype} pen={penalty} k={top_k}")
    pen = {} if penalty == 1.0 else {"penalty": penalty, "history": torch.from_numpy(np.stack(hists)).repeat(rows // 2, 1).to(gpu)}
    got = verify.sample_logits(batch.to(gpu), u.to(gpu), 1.0, top_p, top_k=top_k, **pen)
    res = verify.filter_logits(batch.to(gpu), 1.0, top_p, top_k=top_k) if not pen else None
    torch.cuda.synchronize()
    want = [osmp.filter_row(osmp.process_logits(batch[r].float().numpy(), 1.0, penalty, hists[r] if pen else None,
                                                epv_of(dtype)), top_p, top_k) for r in range(2)]
    assert got.cpu().tolist() == [osmp.categorical_pick(want[r % 2].P, u[r].item()) for r in range(rows)]
    for r in range(rows if res else 0):
        assert res["cutoff"][r].item() == want[r % 2].cutoff, r
        assert res["mass"][r].item() == nm.mass_to_f32(want[r % 2].mass_fx), r
    if res:
        P = torch.from_numpy(np.stack([w.P for w in want])).to(gpu).repeat(rows // 2, 1)
        assert torch.equal(res["filtered"], P)
