"""The calls run on torch's current stream, also inside a stream context and from several threads."""

import threading

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def test_current_stream_of_each_thread():
    from dirktensor_amd import attention as A

    x = torch.zeros(1, device="cuda")
    assert A._stream_of(x) == torch.cuda.current_stream().cuda_stream
    side = [torch.cuda.Stream() for _ in range(2)]
    seen = {}

    def run(i):
        with torch.cuda.stream(side[i]):
            seen[i] = A._stream_of(x)

    ts = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert [seen[i] for i in range(2)] == [s.cuda_stream for s in side]
    with torch.cuda.stream(side[0]):
        assert A._stream_of(x) == side[0].cuda_stream


def test_call_is_ordered_on_the_current_stream():
    from dirktensor_amd import flash_attention_forward

    g = torch.Generator(device="cuda").manual_seed(0)
    q, k, v = (torch.randn((1, 300, 4, 128), generator=g, device="cuda").bfloat16() for _ in range(3))
    want = flash_attention_forward(q, k, v, 0.1, True).output
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        k2 = torch.zeros_like(k)
        for _ in range(20):
            torch.cuda._sleep(100000)
        k2.copy_(k)  # the call has to wait for this
        got = flash_attention_forward(q, k2, v, 0.1, True).output
    s.synchronize()
    assert torch.equal(got, want)
