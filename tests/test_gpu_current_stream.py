"""The Python view's default stream is torch's current one (GPU): inside and
outside a stream context, and in a thread with a stream of its own."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_default_stream_follows_torch(mfx):
    assert mfx._stream(None) == torch.cuda.current_stream().cuda_stream
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert mfx._stream(None) == side.cuda_stream
        seen = []
        t = threading.Thread(target=lambda: seen.append((mfx._stream(None), torch.cuda.current_stream().cuda_stream)))
        t.start()
        t.join()
        assert seen[0][0] == seen[0][1]
    assert mfx._stream(None) == torch.cuda.current_stream().cuda_stream
