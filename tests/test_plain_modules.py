"""Which modules MosAttention's training kernels may stand for: a module that
anything hooks or overrides is called instead."""
import pytest
import torch
from torch import nn

from ssla_amd.layers import _plain_linear, _plain_norm


def _hook(*_):
    return None


@pytest.mark.parametrize("make,plain", [
    (lambda: nn.Linear(8, 12, bias=False), _plain_linear),
    (lambda: nn.LayerNorm(12), lambda m: _plain_norm(m, 12, torch.device("cpu"))),
])
def test_plain_modules(make, plain):
    assert plain(make())
    for register in ("register_forward_hook", "register_forward_pre_hook", "register_full_backward_hook",
                     "register_full_backward_pre_hook"):
        m = make()
        handle = getattr(m, register)(_hook)
        assert not plain(m), register
        handle.remove()
        assert plain(m), register
    m = make()
    m.forward = lambda x: x
    assert not plain(m), "a forward on the instance"
    del m.forward
    for register in (nn.modules.module.register_module_forward_hook,
                     nn.modules.module.register_module_forward_pre_hook,
                     nn.modules.module.register_module_full_backward_hook):
        handle = register(_hook)
        try:
            assert not plain(m), register.__name__
        finally:
            handle.remove()
    assert plain(m)
    assert not plain(type("Sub", (type(m),), {})(*((8, 12) if isinstance(m, nn.Linear) else (12,))))
