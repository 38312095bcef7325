"""vec_dot in one launch: bit for bit the quantizer followed by the GEMV (the kernels the oracle
tests pin), over the edges of the fused kernel's row lengths, lane groups and row counts."""
import numpy as np
import pytest
import torch

import jero_hip as J
from qdata import rand_act, rand_weights

pytestmark = pytest.mark.gpu

# n_in: one block; 4, 16, 32 and 64 lanes per row; 2 and 4 units per lane; one block more and less
KQ = [256, 1024, 1280, 2048, 2304, 4096, 4352, 7936, 8192, 8448]
Q32 = [32, 128, 160, 512, 544, 1024, 1056, 2048, 2080, 4064, 4096, 4128, 6176, 8192, 8224]


def both(quant, laid, n_in, n_out, x=None, y=None):
    dev = torch.device("cuda", 0)
    w = J.TensorView("w", quant, [n_in, n_out], torch.from_numpy(rand_weights(quant, n_out, n_in, n_in + n_out)).to(dev))
    if laid:
        w = J.repack(w)
    x = torch.from_numpy(rand_act(n_in, 7)).to(dev) if x is None else x
    ref = torch.empty(n_out, device=dev)
    J.matvec(w, J.quantize_act(J.act_format(w.quant), x), ref)
    y = torch.full((n_out,), float("nan"), device=dev) if y is None else y
    J.matvec_any(y, w, x)
    torch.cuda.synchronize()
    return y.cpu().numpy(), ref.cpu().numpy()


@pytest.mark.parametrize("n_out", [1, 15, 129, 2049, 4097])
@pytest.mark.parametrize("quant,laid", [(J.Q4_K, False), (J.Q4_K, True), (J.Q6_K, False), (J.Q6_K, True),
                                        (J.Q8_0, False), (J.Q4_0, False)])
def test_one_launch_equals_two(quant, laid, n_out):
    for n_in in KQ if quant in (J.Q4_K, J.Q6_K) else Q32:
        y, ref = both(quant, laid, n_in, n_out)
        assert np.array_equal(y.view(np.uint32), ref.view(np.uint32)), n_in


# rows beyond 4096 elements run fused where the workgroups of 16 (or 8) rows leave no short last round
# of the 256 CUs: from 4096 outputs, at whole rounds, and at 500 workgroups with a partial last one
@pytest.mark.parametrize("n_out", [4096, 7999])
@pytest.mark.parametrize("quant,laid,rows", [
    (J.Q4_K, False, [4352, 7936]), (J.Q4_K, True, [4352, 6400, 8192]), (J.Q6_K, True, [4352, 5120]),
    (J.Q8_0, False, [4128, 6176, 8192]), (J.Q4_0, False, [4128, 7168, 8192])])
def test_long_rows(quant, laid, rows, n_out):
    for n_in in rows:
        y, ref = both(quant, laid, n_in, n_out)
        assert np.array_equal(y.view(np.uint32), ref.view(np.uint32)), n_in


@pytest.mark.parametrize("quant,n_in,n_out", [(J.Q4_K, 256, 25000), (J.Q8_0, 128, 400000), (J.Q4_K, 2304, 24577)])
def test_many_rows(quant, n_in, n_out):
    y, ref = both(quant, False, n_in, n_out)
    assert np.array_equal(y.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("quant", [J.Q4_K, J.Q8_0])
def test_zero_nan_and_overlapping_input(quant):
    dev = torch.device("cuda", 0)
    x = torch.zeros(1024, device=dev)
    y, ref = both(quant, False, 1024, 64, x=x)
    assert np.all(y == 0.0) and np.all(ref == 0.0)
    x = torch.from_numpy(rand_act(1024, 3)).to(dev)
    x[5] = float("inf")
    y, ref = both(quant, False, 1024, 64, x=x)
    assert np.array_equal(np.isnan(y), np.isnan(ref))
    buf = torch.from_numpy(rand_act(1536, 4)).to(dev)
    x = buf[:1024]
    _, ref = both(quant, False, 1024, 512, x=x.clone())
    got, _ = both(quant, False, 1024, 512, x=x, y=buf[1000:1512])  # the output's head lies on the input's tail
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
