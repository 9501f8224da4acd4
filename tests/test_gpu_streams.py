"""Every operator call goes to the caller's current stream: the raw handle that the Python layer passes
is that of torch.cuda.current_stream, which is per thread, and a call made on another stream orders with
that stream's work."""
import threading

import pytest

from gpu_util import need_gpu, torch
from moa_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["default", "side", "external", "nested", "thread"])
def test_handle_is_the_current_streams(kind):
    need_gpu()
    t = torch.zeros(8, device="cuda")
    seen = []

    def look():
        seen.append((ops._stream(t), torch.cuda.current_stream().cuda_stream))

    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    if kind == "default":
        look()
    elif kind == "side":
        with torch.cuda.stream(a):
            look()
        look()
    elif kind == "external":
        with torch.cuda.stream(torch.cuda.ExternalStream(a.cuda_stream)):
            look()
        assert seen[0][0] == a.cuda_stream
    elif kind == "nested":
        with torch.cuda.stream(a):
            with torch.cuda.stream(b):
                look()
            look()
        assert [s[0] for s in seen] == [b.cuda_stream, a.cuda_stream]
    else:  # a new thread starts on the default stream, whatever its creator's is
        with torch.cuda.stream(a):
            th = threading.Thread(target=look)
            th.start()
            th.join()
            look()
        assert seen[0][0] != seen[1][0] == a.cuda_stream
    assert seen and all(x == y for x, y in seen)


def test_call_on_a_side_stream_follows_that_streams_work():
    need_gpu()
    g = torch.Generator(device="cuda").manual_seed(5)
    draw = lambda *shape: torch.randn(shape, generator=g, device="cuda").to(torch.bfloat16)
    q, k, v = draw(1, 8, 2, 256), draw(1024, 8, 256), draw(1024, 8, 256)
    mask = torch.ones(1, 1024, device="cuda")
    want, got, late = torch.empty_like(q), torch.empty_like(q), torch.zeros_like(q)
    ops.sliding_attention(q, k, v, mask, want)
    torch.cuda.synchronize()
    big = torch.randn(4096, 4096, device="cuda")
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for _ in range(8):
            big = big @ big * 1e-3  # work of some ms, behind which q arrives
        late.copy_(q)
        ops.sliding_attention(late, k, v, mask, got)
    s.synchronize()
    assert torch.equal(got, want)
