"""The native binding of the linear entries: what it reads from its arguments and which
errors it raises (stand-ins for device tensors, no GPU), and the streams it takes."""
if __name__ == "__main__":  # `python tests/<file>.py`, as the reference runs its tests
    import sys as _sys

    import pytest as _pytest
    _sys.exit(_pytest.main([__file__, "-q"]))
import ctypes

import numpy as np
import pytest
import torch  # before the library: both then share torch's HIP runtime

from jjjetson_ops_amd import capi


class Fake:
    def __init__(self, cuda=True, contiguous=True):
        self.is_cuda, self._c = cuda, contiguous

    def is_contiguous(self):
        return self._c

    def data_ptr(self):
        return 0x1000


@pytest.mark.parametrize("entry", [capi.linear_q4_0, capi.linear_q4_0_split])
def test_linear_binding_errors(entry):
    ok = Fake()
    for bad, text in ((Fake(cuda=False), "must be a device tensor"), (Fake(contiguous=False), "must be contiguous")):
        for k in range(3):
            args = [ok, ok, ok]
            args[k] = bad
            with pytest.raises(ValueError, match=("x", "w", "y")[k] + " " + text):
                entry(*args, 128, 4, 1, stream=0)
        with pytest.raises(ValueError, match="ws " + text):
            entry(ok, ok, ok, 128, 4, 1, ws=bad, stream=0)
    for k in range(3):
        args = [128, 4, 1]
        args[k] = float(args[k])
        with pytest.raises(ctypes.ArgumentError, match=f"argument {6 + k}"):  # as from every other entry
            entry(ok, ok, ok, *args, stream=0)
    with pytest.raises(AttributeError):
        entry(None, ok, ok, 128, 4, 1, stream=0)
    with pytest.raises(capi.JJOError) as e:  # refused before any device is touched
        entry(ok, ok, ok, 128, 0, 1, stream=0)
    assert e.value.code == capi.JJO_ERR_INVALID_ARG and "out_features=0" in str(e.value)


class AsParameter:
    _as_parameter_ = ctypes.c_int(0)


@pytest.mark.parametrize("entry", [capi.linear_q4_0, capi.linear_q4_0_split])
@pytest.mark.parametrize("zero", [np.int64(0), False, 1 << 32, ctypes.c_int(0), AsParameter()])
def test_linear_binding_ints(entry, zero):
    """A size may be whatever ctypes takes for a C int; the entry refuses the zero itself."""
    ok = Fake()
    with pytest.raises(capi.JJOError) as e:
        entry(ok, ok, ok, 128, zero, 1, stream=0)
    assert e.value.code == capi.JJO_ERR_INVALID_ARG and "out_features=0" in str(e.value)


@pytest.mark.gpu
def test_linear_binding_streams(dev):
    """The current stream, a stream object and a raw handle give the same result."""
    from oracle import c_oracle
    K, N = 256, 64
    rng = np.random.default_rng(0)
    w_h = c_oracle.quantize_q4_0((rng.standard_normal((N, K)) * 0.02).astype(np.float32))
    x_h = rng.standard_normal((1, K)).astype(np.float32)
    exp = c_oracle.matmul(w_h, c_oracle.quantize_q8_1(x_h, [K, 1]), K, N, 1)[0]
    w, x = torch.from_numpy(w_h).to(dev), torch.from_numpy(x_h).to(dev)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    for stream in (None, side, side.cuda_stream):
        y = torch.full((N,), float("nan"), device=dev)
        torch.cuda.synchronize()
        capi.linear_q4_0(x, w, y, K, N, 1, stream=stream)
        torch.cuda.synchronize()
        np.testing.assert_allclose(y.cpu().numpy(), exp, rtol=1e-3, atol=1e-4)
    with torch.cuda.stream(side):
        assert capi._current_stream() == side.cuda_stream
