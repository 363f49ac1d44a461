"""Which calls reach an operator's implementations (Operator.register_backend, Operator.__call__)."""

import functools

import pytest

import xlb_amd as xa
from xlb_amd.operator.operator import Operator

BACKEND = xa.ComputeBackend.MI355X


def _operator(name):
    policy = xa.PrecisionPolicy.FP32FP32
    vs = xa.velocity_set.D2Q9(policy, BACKEND)
    xa.init(velocity_set=vs, default_backend=BACKEND, default_precision_policy=policy)
    return type(name, (Operator,), {})


@pytest.mark.parametrize("how", ["wraps", "signature"])
def test_a_decorated_implementation_takes_what_its_signature_says(how):
    """A decorator that takes anything does not run for a call that the signature refuses."""
    ran = []

    def scale(self, f, factor):
        return f * factor

    if how == "wraps":

        @functools.wraps(scale)
        def implementation(self, *args, **kwargs):
            ran.append(args)
            return scale(self, *args[:2])
    else:

        def implementation(self, *args):
            ran.append(args)
            return scale(self, *args[:2])

        import inspect

        implementation.__signature__ = inspect.signature(scale)
    cls = _operator("ScaleBy" + how)
    implementation.__qualname__ = f"{cls.__name__}.implementation"
    cls.register_backend(BACKEND)(implementation)
    assert cls()(2, 3) == 6 and len(ran) == 1
    with pytest.raises(Exception, match="too many positional"):
        cls()(2, 3, 4)
    assert len(ran) == 1


def test_an_implementation_registered_during_a_look_up_is_found_by_the_next_call():
    """As when another thread imports the module that registers it."""
    cls = _operator("AddUp")

    def register(func):
        func.__qualname__ = "AddUp.implementation"
        cls.register_backend(BACKEND)(func)

    class Table(dict):
        late = None

        def items(self):
            seen = list(super().items())
            if self.late is not None:
                late, self.late = self.late, None
                register(late)
            return seen

    cls._backends, cls._signatures = Table(), {}
    register(lambda self, a: a)
    cls._backends.late = lambda self, a, b: a + b
    with pytest.raises(Exception):
        cls()(1, 2)
    assert cls()(1, 2) == 3
