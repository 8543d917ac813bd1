"""The autograd layer's calls go to the device that the tensors are on, whichever is
the current one: device index and stream of the energy hooks, and the streams that
library calls are ordered against. On the CPU, with stand-ins for tensors of a second
device and for torch.cuda while the first one is current."""
from types import SimpleNamespace

import pytest

torch = pytest.importorskip("torch")
autograd = pytest.importorskip("spfft_amd.autograd")

CURRENT, OTHER = torch.device("cuda", 0), torch.device("cuda", 1)


class Tensor:
    """What the layer asks of a tensor of two bands of 3 x 4 x 5 on `OTHER`."""

    def __init__(self, dtype, shape):
        self.dtype, self.shape, self.device = dtype, torch.Size(shape), OTHER
        self.requires_grad = False

    def data_ptr(self):
        return 4096

    def element_size(self):
        return 8

    def numel(self):
        return self.shape.numel()

    def is_contiguous(self):
        return True

    def is_neg(self):
        return False

    is_conj = is_neg


@pytest.fixture
def calls(monkeypatch):
    made = []

    def hook(name):
        return lambda *args: made.append((name, args)) or 0

    def stream(kind):
        def of(device=None):
            index = 0 if device is None else torch.device(device).index
            return SimpleNamespace(cuda_stream=(10 if kind == "current" else 20) + index,
                                   wait_stream=lambda s: made.append((kind, index, s.cuda_stream)))
        return of

    for name in ("spfft_amd_field_energy", "spfft_amd_energy_field"):
        monkeypatch.setattr(autograd.sp.lib, name, hook(name))
    monkeypatch.setattr(autograd.torch, "empty",
                        lambda *a, dtype=None, device=None: Tensor(dtype, a[0] if a else ()) if
                        isinstance(a[0], tuple) else Tensor(dtype, (a[0],)))
    monkeypatch.setattr(autograd.torch, "empty_like", lambda x: Tensor(x.dtype, x.shape))
    monkeypatch.setattr(autograd.torch.cuda, "current_stream", stream("current"))
    monkeypatch.setattr(autograd.torch.cuda, "default_stream", stream("default"))
    monkeypatch.setattr(autograd, "_batch_adjoint", lambda transforms, n, field: field)
    return made


def test_energy_hooks_name_the_tensors_device_and_stream(calls):
    psi, potential = Tensor(torch.complex128, (2, 3, 4, 5)), Tensor(torch.float64, (3, 4, 5))
    autograd._band_energy(psi, potential)
    autograd._energy_gradient([SimpleNamespace(num_values=7)], psi, False, potential,
                              Tensor(torch.float64, ()))
    assert [name for name, _ in calls] == ["spfft_amd_field_energy", "spfft_amd_energy_field"]
    for _, args in calls:
        assert args[0] == OTHER.index and args[-1] == 10 + OTHER.index


def test_library_calls_are_ordered_on_the_tensors_device(calls):
    with autograd._OnDefaultStream(OTHER):
        pass
    assert calls == [("default", 1, 11), ("current", 1, 21)]
