"""What tensor_context binds, and that it binds it once."""
import pytest

from cortex_amd import tensor as ct


def bound():
    return ct._stream.get(None), ct._datatype.get(None)


def test_a_context_entered_again_is_refused_and_the_binding_restored():
    before = bound()
    context = ct.tensor_context("stream", "float")
    with context:
        with pytest.raises(RuntimeError):
            context.__enter__()
        assert bound() == ("stream", "float")
    assert bound() == before
    with pytest.raises(RuntimeError):
        context.__enter__()
    assert bound() == before


def test_nested_contexts_and_decorated_functions():
    before = bound()

    @ct.tensor_context("outer", "double")
    def depth(n):
        assert bound() == ("outer", "double")
        with ct.tensor_context(n, "float") as stream:
            assert stream == n and bound() == (n, "float")
            if n:
                depth(n - 1)
            assert bound() == (n, "float")

    depth(2)
    depth(1)
    assert bound() == before
