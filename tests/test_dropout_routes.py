"""Which buffers the dropout layer gives to a driver's one-launch mask.  The launch takes whole float or double
multipliers, float draws and one count for both; everything else belongs to the chain of tensor calls."""
import numpy as np
import pytest

import oracle_backend
from cortex_amd import nn_layers as layers
from cortex_amd import tensor as ct


class Asked(Exception):
    pass


def layer_on(datatype, fused):
    device = oracle_backend.OracleDriver().default_device()
    stream = oracle_backend.OracleStream(device)
    if fused:
        def mask(mult_buffer, rand_buffer, probability):
            raise Asked
        stream.dropout_bernoulli_mask = mask
    stream.seed_random(5)
    with ct.tensor_context(stream, "float"):
        layer = layers.create({"type": "dropout", "distribution": "bernoulli", "probability": 0.5, "input-size": 6}, 4,
                              datatype)
    return stream, layer


@pytest.mark.parametrize("datatype", ["float", "double"])
def test_float_multipliers_take_one_launch(datatype):
    stream, layer = layer_on(datatype, True)
    with ct.tensor_context(stream, "float"), pytest.raises(Asked):
        layer.prepare_forward()


@pytest.mark.parametrize("datatype", ["int", "long", "short", "byte"])
def test_integer_multipliers_take_the_chain(datatype):
    got = []
    for fused in (False, True):
        stream, layer = layer_on(datatype, fused)
        with ct.tensor_context(stream, "float"):
            layer.prepare_forward()
            got.append(ct.to_double_array(layer.mult_buffer))
    assert np.array_equal(*got)


def test_draws_of_another_count_take_the_chain():
    """One row of draws under four of multipliers: the chain spreads them, the launch would write past their end."""
    got = []
    for fused in (False, True):
        stream, layer = layer_on("double", fused)
        with ct.tensor_context(stream, "float"):
            layer.rand_buffer = ct.new_tensor([1, 6], datatype="float")
            layer.prepare_forward()
            got.append(ct.to_double_array(layer.mult_buffer))
    assert np.array_equal(*got) and np.array_equal(got[0].reshape(4, 6)[0], got[0].reshape(4, 6)[3])
