"""The d_model-64 persistent decode loads each phase's weights, and the next
layer's or the head's, ahead of it: one layer (no next layer) and two, one
lane, a block and a lane more, with a short last chunk, give the oracle's
container bytes and a byte-identical round trip."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers", [1, 2])
@pytest.mark.parametrize("lanes", [1, 4, 5, 1029])
def test_layers_and_lanes(oracle, make_weights, layers, lanes):
    import torch

    import boa_hip
    w = make_weights(64, layers, 16)
    chunk = 19
    data = np.random.default_rng(lanes).integers(0, 256, lanes * chunk - 3, dtype=np.uint8).tobytes()
    c = boa_hip.Codec(64, layers, 16, lanes, 0, 1.0)
    c.set_stream(torch.cuda.current_stream().cuda_stream)
    c.load_weights(w)
    assert c.decode_plan(lanes)["persistent"]
    blob = c.compress(data, chunk_size=chunk)
    assert blob == oracle.Model(w, 64, layers).compress(data, chunk_size=chunk)
    assert c.decompress(blob) == data
    c.close()
