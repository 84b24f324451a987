"""The CPython extension on the CPU: what torch throws inside it arrives as a Python exception."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from blockgtq_amd import _host


def _cache(B=1, n_kv=1, T=64):
    u8, f16 = dict(dtype=torch.uint8, device="cuda"), dict(dtype=torch.float16, device="cuda")
    return [torch.empty(1024, **u8), torch.empty(B, n_kv, T, 52, **u8), torch.empty(B, n_kv, T, 5, **f16),
            torch.empty(B, n_kv, T, 48, **u8), torch.empty(B, n_kv, T, **f16)]


@pytest.mark.skipif(torch.cuda.is_available(), reason="without a GPU, so that nothing is ever launched")
@pytest.mark.filterwarnings("ignore:Accessing the data pointer")
@pytest.mark.parametrize("entry", ["step", "encode", "attend", "prompt"])
def test_torch_errors_arrive_as_exceptions(entry):
    mod = _host.module()
    with FakeTensorMode(allow_non_fake_inputs=True):        # GPU tensors with shapes and no memory
        plans, kp, kn, vp, vn = _cache()
        q = torch.empty(1, 4, 1, 128, dtype=torch.float16, device="cuda")
        k = torch.empty(1, 1, 1, 128, dtype=torch.float16, device="cuda")
    class Ws:
        _buf = None

    def layer():
        return mod.Layer(plans, kp, kn, vp, vn, 52, 5, 48, 4, 0, 0, 0.1, False, None, None)

    with pytest.raises(RuntimeError):
        if entry == "step":
            layer().step(q, k, k, 3, 4, None, 1, 0, Ws())
        elif entry == "encode":
            layer().encode(k, k, 3, 0)
        elif entry == "attend":
            mod.attend(plans, q, kp, kn, vp, vn, 64, 1, 0, 0, 0.1, 1, Ws())
        else:
            mod.prompt(plans, q, 1, kp, kn, vp, vn, 64, 52, 48, 0, 1, 0, 0, 0.1, 1)
