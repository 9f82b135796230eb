"""The stream a call without one runs on: torch's current stream, under the
default stream, a stream context, a nested one and another thread."""
import threading

import pytest

import kvbridge_amd as kvb

pytestmark = pytest.mark.gpu


def test_current_stream_is_torchs(gpu):
    import torch

    def same():
        assert kvb._stream(None) == torch.cuda.current_stream().cuda_stream

    same()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(a):
        same()
        assert kvb._stream(None) == a.cuda_stream
        with torch.cuda.stream(b):
            assert kvb._stream(None) == b.cuda_stream
            seen = []
            t = threading.Thread(target=lambda: seen.append((kvb._stream(None), torch.cuda.current_stream().cuda_stream)))
            t.start()
            t.join()
            assert seen[0][0] == seen[0][1]
        same()
    assert kvb._stream(a) == a.cuda_stream and kvb._stream(5) == 5
