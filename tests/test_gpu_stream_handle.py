"""The front end's stream argument: the current stream's handle, also where torch lacks the private
names that it is read by."""
import pytest
import torch

import jero_hip as J

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("private", [True, False])
def test_current_stream_handle(dev, monkeypatch, private):
    side = torch.cuda.Stream()
    monkeypatch.setattr(J, "_raw_stream", None)
    with monkeypatch.context() as m:
        if not private:
            m.delattr(torch._C, "_cuda_getCurrentRawStream")
        J._stream()  # chooses the way
    for _ in range(2):
        assert J._stream() == torch.cuda.current_stream().cuda_stream
        with torch.cuda.stream(side):
            assert J._stream() == side.cuda_stream
    assert J._stream(side) == side.cuda_stream
