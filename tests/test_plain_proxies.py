"""A module that passes itself off as the class it wraps is still called (no GPU: only the choice)."""
from torch import nn

from nano_vllm_x_amd.layers import plain


class Proxy:
    """Hands every look-up on, that of its class and of its dictionary among them, and counts calls."""

    def __init__(self, inner):
        object.__setattr__(self, "_inner", inner)

    def __getattribute__(self, name):
        return getattr(object.__getattribute__(self, "_inner"), name)

    def __call__(self, *args):
        return 0.5 * object.__getattribute__(self, "_inner")(*args)


def test_a_proxy_is_not_the_module_inside():
    m = nn.Linear(4, 4, bias=False)
    p = Proxy(m)
    assert isinstance(p, nn.Linear) and p.__class__ is nn.Linear
    assert plain.untouched(m, nn.Linear) and not plain.untouched(p, nn.Linear)
