"""The GEMM's few-token form (K split over a workgroup's waves) and the Q4_K kernel at rows that are not
a multiple of its tile, against one GEMV per row (held to the oracle by the GEMV tests).  Both sum
the same exact block terms in f32 in another order: nb terms of at most the row's magnitude differ
by a few nb * 2^-24, below 1e-5 of it for the 57 blocks here at most."""
import numpy as np
import pytest
import torch

import jero_hip as J
from qdata import rand_act, rand_weights

pytestmark = pytest.mark.gpu


def check(quant, laid, m, n_in, n_out):
    dev = torch.device("cuda", 0)
    w = J.TensorView("w", quant, [n_in, n_out], torch.from_numpy(rand_weights(quant, n_out, n_in, n_in + n_out)).to(dev))
    x = torch.from_numpy(rand_act(m * n_in, m)).view(m, n_in).to(dev)
    xq = J.quantize_act(J.Q8_K, x)
    y = torch.full((m + 1, n_out), 7.0, device=dev)
    J.gemm(J.repack_gemm(w) if laid else w, xq, m, y)
    ref = torch.empty(m, n_out, device=dev)
    for r in range(m):
        J.matvec(w, xq.view(m, -1)[r].contiguous(), ref[r])
    torch.cuda.synchronize()
    got, want = y.cpu().numpy(), ref.cpu().numpy()
    scale = np.maximum(np.abs(want), np.sqrt(np.mean(want ** 2)))
    assert np.all(np.abs(got[:m] - want) <= 1e-5 * scale)
    assert np.all(got[m] == 7.0)  # nothing past the last row


# tiles: one, up to a CU each (eight waves), above it (four waves), and past the rule's end
@pytest.mark.parametrize("m,n_out", [(1, 32), (8, 1000), (31, 64), (33, 4096), (64, 8192), (100, 31), (96, 8224)])
@pytest.mark.parametrize("n_in", [256, 1792, 2304, 12288])  # fewer blocks than waves; ragged runs
@pytest.mark.parametrize("quant", [J.Q4_K, J.Q6_K])
def test_few_tokens(quant, n_in, m, n_out):
    check(quant, True, m, n_in, n_out)


# both sides of the rules between the forms: one block of K (two and more tiles per CU), records of 68
# and 72 MB, and K halves within the workgroup or over the grid by the row's length and the tiles
@pytest.mark.parametrize("quant,n_in,m,n_out", [
    (J.Q4_K, 256, 128, 4096), (J.Q4_K, 256, 129, 4096), (J.Q6_K, 256, 97, 8192), (J.Q6_K, 8192, 161, 4096),
    (J.Q6_K, 8704, 161, 4096), (J.Q4_K, 14336, 129, 4096), (J.Q6_K, 6144, 257, 4096), (J.Q6_K, 6400, 257, 4096),
    (J.Q6_K, 6400, 449, 4096), (J.Q4_K, 14592, 257, 4096)])
def test_rule_edges(quant, n_in, m, n_out):
    check(quant, True, m, n_in, n_out)


@pytest.mark.parametrize("laid_rows", [False, True])
@pytest.mark.parametrize("m,n_out,n_in", [(15, 96, 1024), (16, 96, 1024), (17, 31, 1024), (130, 1000, 1024),
                                          (129, 4100, 1024), (29, 96, 12288), (30, 96, 12288), (16, 2080, 12288)])
def test_ragged_rows(m, n_out, n_in, laid_rows):
    if laid_rows:
        dev = torch.device("cuda", 0)
        w = J.TensorView("w", J.Q4_K, [n_in, n_out], torch.from_numpy(rand_weights(J.Q4_K, n_out, n_in, 5)).to(dev))
        x = J.quantize_act(J.Q8_K, torch.from_numpy(rand_act(m * n_in, m)).view(m, n_in).to(dev))
        a, b = torch.empty(m, n_out, device=dev), torch.empty(m, n_out, device=dev)
        J.gemm(w, x, m, a)
        J.gemm(J.repack(w), x, m, b)
        torch.cuda.synchronize()
        assert torch.equal(a, b)
    else:
        check(J.Q4_K, False, m, n_in, n_out)
