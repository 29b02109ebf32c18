"""Zeroing by the library's kernel: sizes around a word, a thread's words, a
workgroup's and the size where the stores go past the caches, with the bytes
on both sides untouched; and the tensors that torch's zero_ has to take."""
import numpy as np
import pytest

from pyop2_amd import device as dev, op2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbytes", [0, 1, 8, 15, 16, 17, 4095, 4096, 4097, 16383, 16384, 16385, 16400, 1000003,
                                    (256 << 20) - 1, 256 << 20, (256 << 20) + 1, (256 << 20) + 4113])
def test_bytes(device, nbytes):
    torch = dev.torch()
    whole = torch.full((nbytes + 64,), 7, dtype=torch.uint8, device=dev.device())
    for at in (16, 32):
        whole.fill_(7)
        part = whole[at:at + nbytes]
        version = part._version
        dev.clear(part)
        assert part._version > version
        assert not part.any() and (whole[:at] == 7).all() and (whole[at + nbytes:] == 7).all()


def test_other_tensors(device):
    torch = dev.torch()
    base = torch.ones(20, 6, dtype=torch.float64, device=dev.device())
    dev.clear(base[:, 1:3])          # strided
    assert base.sum() == 80 and not base[:, 1:3].any()
    flat = torch.ones(9, dtype=torch.float64, device=dev.device())
    dev.clear(flat[1:8])             # not on a 16-byte boundary
    assert flat.tolist() == [1.0] + [0.0] * 7 + [1.0]
    leaf = torch.ones(4, dtype=torch.float64, device=dev.device(), requires_grad=True)
    with pytest.raises(RuntimeError):
        dev.clear(leaf)
    with torch.no_grad():
        dev.clear(leaf)
    assert not leaf.any()
    with torch.inference_mode():
        t = torch.ones(4, device=dev.device())
        dev.clear(t)
        assert not t.any()


def test_zero_in_a_captured_graph(device):
    torch = dev.torch()
    s = op2.Set(1000)
    d = op2.Dat(s ** 3, np.ones((1000, 3)))
    t = d.device_data
    d.zero()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        d.zero()
        d.device_data.add_(2.0)
    for _ in range(3):
        t.fill_(5.0)
        graph.replay()
        assert (t == 2.0).all()
