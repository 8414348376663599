"""The Python binding's fast paths: the current stream it passes, and the tensor
checks that a fitting tensor passes in one expression."""
from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu


def test_current_stream(hip, torch_gpu):
    torch = torch_gpu
    side = torch.cuda.Stream()
    assert hip._stream() == torch.cuda.current_stream().cuda_stream
    with torch.cuda.stream(side):
        assert hip._stream() == side.cuda_stream
    assert hip._stream(side) == side.cuda_stream


@pytest.mark.parametrize("bad", ["host", "strided", "short"])
@pytest.mark.parametrize("which", ["activation", "weight", "out", "workspace"])
def test_checks(hip, torch_gpu, which, bad):
    torch = torch_gpu
    m, n, k = 3, 64, 256
    size = {"activation": (m, k * 4), "weight": (n, k // 32 * 18), "out": (m, n * 4), "workspace": (m, k // 32 * 34)}
    kinds = {"activation": torch.float32, "out": torch.float32}
    made = {name: torch.zeros(shape, dtype=torch.uint8, device="cuda").view(kinds.get(name, torch.uint8))
            for name, shape in size.items()}
    t = made[which]
    made[which] = {"host": t.cpu(), "strided": torch.cat([t, t], 1)[:, ::2],
                   "short": t[:, :-1].contiguous() if which != "activation" else t.to(torch.float16)}[bad]
    with pytest.raises(ValueError, match=which):
        hip.compute(hip.Q4_0, made["activation"], made["weight"], n, out=made["out"], workspace=made["workspace"])
