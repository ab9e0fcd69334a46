"""The dropout layer through the driver's one-launch mask and through the chain of tensor calls: the same multipliers,
draws and generator state."""
import numpy as np
import pytest

from cortex_amd import driver as drv
from cortex_amd import nn_layers as layers
from cortex_amd import tensor as ct

pytestmark = pytest.mark.gpu


class ChainStream(drv.HipStream):
    dropout_bernoulli_mask = None


@pytest.mark.parametrize("datatype", ["float", "double"])
@pytest.mark.parametrize("batch,items", [(1, 2), (3, 5), (128, 128)])
@pytest.mark.parametrize("probability", [0.8, 1.0, 1e-3])
def test_one_launch_mask_is_the_chain(datatype, batch, items, probability):
    device = drv.HipDriver().default_device()
    drawn = []
    for kind in (drv.HipStream, ChainStream):
        stream = kind(device, None)
        stream.seed_random(17)
        with ct.tensor_context(stream, datatype):
            layer = layers.create({"type": "dropout", "distribution": "bernoulli", "probability": probability,
                                   "input-size": items}, batch, datatype)
            got = []
            for _ in range(2):      # the second draw starts where the first left the generator
                layer.prepare_forward()
                got += [ct.to_double_array(layer.mult_buffer), ct.to_double_array(layer.rand_buffer)]
            for t in {id(t): t for t in (layer.mult_buffer, layer.rand_buffer)}.values():
                t.buffer.release()
        drawn.append(got)
    for one, chain in zip(*drawn):
        assert np.array_equal(one, chain)
