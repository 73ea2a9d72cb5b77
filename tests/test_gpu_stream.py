"""The stream that a call is given is torch's current one: by default, inside a
stream context and after it, in another thread and in a capture."""
import threading

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from gpt_amd import core  # noqa: E402


def same():
    return (core.stream_ptr() or 0) == torch.cuda.current_stream().cuda_stream


def test_the_current_stream():
    side, other = torch.cuda.Stream(), torch.cuda.Stream()
    assert same()
    with torch.cuda.stream(side):
        assert same() and core.stream_ptr() == side.cuda_stream
        with torch.cuda.stream(other):
            assert same()
        seen = []
        t = threading.Thread(target=lambda: seen.append((core.stream_ptr() or 0, same())))
        t.start()
        t.join()
        assert seen == [(torch.cuda.default_stream().cuda_stream, True)]
        assert same()
    assert same()
    x = torch.zeros(8, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ok = same()
        x += 1
    assert ok and same()
