"""Attention of few positions, where the partial kernel writes the output itself, against 64-bit
attention: f32 sums of at most 64 terms around an exponential of relative error |x| 6e-8."""
import numpy as np
import pytest
import torch

import decode_parity as DP
import jero_hip as J
import model_spec as MS
import pyoracle as O
from test_gpu_decode import make_gpu_model, prefill_kv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv", [torch.float16, torch.float32])
@pytest.mark.parametrize("heads,kv_heads,hd", [(32, 8, 128), (8, 8, 64), (16, 2, 128), (4, 4, 32), (6, 2, 64)])
def test_few_positions(heads, kv_heads, hd, kv):
    g = torch.Generator(device="cuda").manual_seed(heads + hd)
    for seq in (1, 2, 15, 16, 17, 63, 64, 65, 129):  # both sides of one split
        q = torch.randn(heads * hd, generator=g, device="cuda")
        k, v = (torch.randn(seq, kv_heads * hd, generator=g, device="cuda").to(kv) for _ in range(2))
        out = torch.full((heads * hd + 8,), 7.0, device="cuda")
        J.gqa_causal_attention_f32(out, q, k, v, heads, kv_heads, hd, seq, 1 / hd ** 0.5)
        torch.cuda.synchronize()
        q64, k64, v64 = q.double().view(heads, hd), k.double().view(seq, kv_heads, hd), v.double().view(seq, kv_heads, hd)
        rep = heads // kv_heads
        p = torch.softmax(torch.stack([k64[:, h // rep] @ q64[h] for h in range(heads)]) / hd ** 0.5, 1)
        ref = torch.stack([p[h] @ v64[:, h // rep] for h in range(heads)]).reshape(-1)
        err = (out[:-8].double() - ref).norm() / ref.norm()
        assert float(err) < 5e-6, (seq, float(err))
        assert np.all(out[-8:].cpu().numpy() == 7.0)


def test_output_over_the_queries():
    g = torch.Generator(device="cuda").manual_seed(3)
    buf = torch.randn(4096 + 128, generator=g, device="cuda")
    k, v = (torch.randn(40, 1024, generator=g, device="cuda").half() for _ in range(2))
    want = torch.empty(4096, device="cuda")
    J.gqa_causal_attention_f32(want, buf[:4096].clone(), k, v, 32, 8, 128, 40, 0.1)
    J.gqa_causal_attention_f32(buf[128:], buf[:4096], k, v, 32, 8, 128, 40, 0.1)
    torch.cuda.synchronize()
    assert torch.equal(buf[128:], want)


@pytest.mark.parametrize("nq,nkv,hd,kv_f16", [(8, 2, 64, False), (4, 2, 128, False), (8, 8, 32, False), (8, 2, 32, True)])
def test_batch_of_queries(dev, nq, nkv, hd, kv_f16):
    """A prompt whose queries all see at most one split of positions, on rings that the flash kernel does
    not take: every query's row lands at its own place (each token against the oracle)."""
    spec = dict(hidden=512, ffn=1024, n_layers=2, vocab=1000, nq=nq, nkv=nkv, hd=hd, eps=1e-6, theta=1e6)
    cap, pos0, n = 128, 5, 40
    t = MS.build(spec, seed=37)
    m = make_gpu_model(spec, t, cap, J.KV_F16 if kv_f16 else J.KV_F32, True)
    om = O.DecodeModel(spec, MS.oracle_tensors(t), cap)
    kv = prefill_kv(m, om, spec, cap, pos0, 41, dev, kv_f16)
    tokens = np.random.default_rng(hd).integers(0, spec["vocab"], size=n).tolist()
    DP.run_prefill_traced(m, om, t, spec, kv, cap, pos0, tokens, kv_f16, dev, True)
    m.close()
