"""evaluate's one-launch decode against single-token forward calls (held to the oracle bit for bit by
the forward tests): the tokens, and the caches it leaves."""
import threading

import numpy as np
import pytest
import torch

import jero_hip as J

pytestmark = pytest.mark.gpu


def expect(seed, vocab, cap, prompt, max_tokens):
    m = J.ForwardModel(seed, vocab, cap)
    logits = torch.empty(max(vocab, 1) + 7, dtype=torch.int32, device="cuda")
    m.forward(prompt, 0, logits)
    out = []
    for i in range(max_tokens):
        torch.cuda.synchronize()
        out.append(int(np.argmax(logits[:max(vocab, 1)].cpu().numpy())))
        if i + 1 < max_tokens:
            m.forward([out[-1]], len(prompt) + i, logits)
    return m, out, logits


def prompt_of(seed, vocab, n):
    return [int(t) for t in np.random.default_rng(seed).integers(0, max(vocab, 1), n)]


# one head row; several reads of the logits and passes of the head; the last position of the launch's
# own rows (need = 128), one more (the graph), one prompt row, one or two K / V blocks, one token; a
# large head before and after a prompt of one K / V block
@pytest.mark.parametrize("vocab,n,max_tokens", [(0, 1, 2), (1, 3, 5), (5, 2, 1), (256, 1, 128), (256, 1, 129), (300, 64, 65),
                                                (777, 60, 8), (4096, 5, 4), (4097, 5, 4), (4096, 64, 3),
                                                (2049, 65, 3), (2048, 65, 3)])
def test_evaluate_equals_forward(vocab, n, max_tokens):
    cap = n + max_tokens
    prompt = prompt_of(n, vocab, n)
    ref, want, logits = expect(99, vocab, cap, prompt, max_tokens)
    m = J.ForwardModel(99, vocab, cap)
    assert m.decode_form == m.DECODE_NONE
    launch = max_tokens > 1 and n + max_tokens - 1 <= 128 and vocab <= (4096 if n <= 64 else 2048)
    for _ in range(2):  # the exchange's words carry on
        assert m.evaluate(prompt, max_tokens) == want
        assert m.decode_form == (m.DECODE_LAUNCH if launch else m.DECODE_GRAPH)
    got = torch.empty_like(logits)
    ref.forward([want[-1]], n + max_tokens - 1, logits)
    m.forward([want[-1]], n + max_tokens - 1, got)
    torch.cuda.synchronize()
    k = max(vocab, 1)
    assert torch.equal(got[:k], logits[:k])


@pytest.mark.parametrize("vocab,n,max_tokens", [(1, 3, 5), (256, 11, 53), (4096, 5, 4)])
def test_waits_in_vain_end_in_the_graph(vocab, n, max_tokens):
    """With no read allowed every wave gives up at once (and leaves the kernel normally); with one a
    step, most do.  Either way the tokens and the caches are those of the graph, and a later evaluate
    runs in one launch again."""
    cap = n + max_tokens
    prompt = prompt_of(n, vocab, n)
    ref, want, logits = expect(99, vocab, cap, prompt, max_tokens)
    ref.forward([want[-1]], n + max_tokens - 1, logits)
    m = J.ForwardModel(99, vocab, cap)
    got = torch.empty_like(logits)
    for polls, forms in ((0, [m.DECODE_TIMED_OUT]), (1, [m.DECODE_TIMED_OUT, m.DECODE_LAUNCH]),
                         (1 << 19, [m.DECODE_LAUNCH]), (0, [m.DECODE_TIMED_OUT]), (1 << 20, [m.DECODE_LAUNCH])):
        m.set_decode_polls(polls)
        assert m.evaluate(prompt, max_tokens) == want, polls
        assert m.decode_form in forms, polls
        m.forward([want[-1]], n + max_tokens - 1, got)
        torch.cuda.synchronize()
        assert torch.equal(got[:max(vocab, 1)], logits[:max(vocab, 1)]), polls


def test_shapes_in_turn_and_two_threads():
    shapes = [(11, 20), (3, 40), (30, 2)]
    want = [expect(5, 256, 64, prompt_of(i, 256, n), k)[1] for i, (n, k) in enumerate(shapes)]
    bad = []

    def work():
        J.init(0)
        m = J.ForwardModel(5, 256, 64)
        s = torch.cuda.Stream()
        for r in range(6):
            i = r % 3
            if m.evaluate(prompt_of(i, 256, shapes[i][0]), shapes[i][1], stream=s) != want[i]:
                bad.append(i)

    threads = [threading.Thread(target=work) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
