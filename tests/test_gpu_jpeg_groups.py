"""The JPEG kernels at the edges of their groups of 4 MCUs (a last group of 1 to 4, groups
that wrap over MCU rows), with dummy blocks at the right and bottom edge, and over the
range of coded lengths (flat frames, full-range noise at quality 100): files and frame
messages equal the oracle's byte for byte."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (height, width): 1, 2, 3, 4, 5 MCUs; odd rows and columns of blocks; 8 x 9 MCUs
SHAPES = [(1, 1), (2, 17), (9, 40), (8, 57), (25, 24), (16, 80), (31, 129), (121, 143), (72, 200)]


def _frames(h, w):
    rng = np.random.default_rng(100 * h + w)
    noise = rng.integers(0, 256, (h, w, 4), dtype=np.uint8)
    edges = (rng.integers(0, 2, (h, w, 4)) * 255).astype(np.uint8)  # saturated: long codes
    ramp = np.minimum(np.add.outer(np.arange(h), np.arange(w))[..., None] * np.array([1, 2, 3, 1]), 255).astype(np.uint8)
    return {"flat": np.full((h, w, 4), 200, np.uint8), "noise": noise, "edges": edges, "ramp": ramp}


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("quality", [1, 60, 100])
def test_files_and_messages_equal_the_oracle(gpu, oracle_lib, shape, quality):
    import torch

    from isaac_amd import frame as K
    from oracle import jpeg_oracle as J

    for name, rgba in _frames(*shape).items():
        dev = torch.from_numpy(rgba).to(gpu)
        want = J.encode(rgba, quality)
        got = K.jpeg(dev, quality)
        print(f"{shape} q{quality} {name}: {len(got)} bytes", flush=True)
        assert got == want, name
        assert K.jpeg_frame_message(dev, quality) == J.frame_message(rgba, quality), name


def test_message_capacity(gpu, oracle_lib):
    """A message buffer too small reports the length, writes nothing and fails."""
    import ctypes

    import torch

    from isaac_amd._lib import lib
    from oracle import jpeg_oracle as J

    L = lib()
    rgba = _frames(33, 50)["noise"]
    dev = torch.from_numpy(rgba).to(gpu)
    want = J.frame_message(rgba, 90)
    nbytes = int(L.isaac_hip_jpeg_workspace_bytes(50, 33))
    ws = torch.empty(nbytes, dtype=torch.uint8, device=gpu)
    buf = ctypes.create_string_buffer(b"x" * 64, len(want) + 1)
    n = ctypes.c_int64(0)
    for cap in (0, len(want), len(want) + 1):
        rc = L.isaac_hip_jpeg_frame_message(ctypes.c_void_p(dev.data_ptr()), 50, 33, 90, ctypes.c_void_p(ws.data_ptr()), nbytes,
                                            buf, cap, ctypes.byref(n), ctypes.c_void_p(0))
        assert n.value == len(want)
        assert (rc == 0) == (cap > len(want))
        if rc:
            assert buf.raw[:64] == b"x" * 64
    assert buf.value == want
