"""Selective scan and activations away from ordinary arguments.

The fp32 kernels run a wave without clamps and selects where every lane's
softplus and gate arguments lie within +-87 and its decay exponents stay
above -126, and through the general forms otherwise.  These weights put
tokens of one wave on both sides of each limit: softplus arguments to +-130,
gate and conv arguments past +-88, decay coefficients from 2^-7 to 2^9 (one
channel far beyond), GELU arguments past the tanh's saturation.  Logits of
every form (token-blocked and scalar-load chunk scan, decode step) equal the
oracle's bit for bit."""
import numpy as np
import pytest

import synth

pytestmark = pytest.mark.gpu


def _extreme_weights(path, d, ds):
    rng = np.random.default_rng(100 + d)
    out = []
    for name, a in synth.random_weight_tensors(d, 1, ds, seed=3):
        a = a.copy()
        if name.endswith("dt_proj.bias"):
            a = rng.uniform(-130, 130, a.shape).astype(np.float32)
            a[::3] = rng.uniform(-3, 3, a[::3].shape)
        elif name.endswith("A_log"):
            a = rng.uniform(-5, 6, a.shape).astype(np.float32)
            a[1] = 20.0
        elif name.endswith("in_proj.weight"):
            a *= rng.choice([1.0, 60.0], size=(a.shape[0], 1)).astype(np.float32)
        elif name.endswith("ff.0.weight"):
            a *= 20
        out.append((name, a))
    synth.write_weights(str(path), out)


@pytest.mark.parametrize("d", [64, 80, 256])
def test_scan_limits_match_the_oracle(oracle, tmp_path, d):
    import torch

    import boa_hip
    w = tmp_path / "w.bin"
    _extreme_weights(w, d, 16)
    T, few = 7, 3
    many = -(-64 * 1024 // (2 * d))  # the first lane count on the scalar-load scan
    tok = np.random.default_rng(d).integers(0, 256, size=(many, T), dtype=np.uint8)
    want = oracle.Model(w, d, 1, 16).new_state(many).forward_chunk(tok)
    for lanes in (few, many):
        c = boa_hip.Codec(d, 1, 16, lanes)
        c.set_stream(torch.cuda.current_stream().cuda_stream)
        c.load_weights(w)
        c.reset_state(lanes)
        got = torch.zeros((lanes, T, 256), device="cuda")
        c.forward_chunk(torch.from_numpy(tok[:lanes].copy()).cuda(), lanes, T, got)
        torch.cuda.synchronize()
        assert np.array_equal(got.cpu().numpy().view(np.uint32), want[:lanes].view(np.uint32))
        c.reset_state(lanes)
        step = torch.zeros((lanes, 256), device="cuda")
        for t in range(T):
            c.step_batch(torch.from_numpy(tok[:lanes, t].copy()).cuda(), lanes, step)
            torch.cuda.synchronize()
            assert np.array_equal(step.cpu().numpy().view(np.uint32),
                                  want[:lanes, t].view(np.uint32)), f"{lanes} lanes, step {t}"
        c.close()


@pytest.mark.parametrize("d,lanes", [(64, 5), (64, 2100), (256, 2100)])
def test_decode_limits_match_the_oracle(oracle, tmp_path, d, lanes):
    """The persistent decode (d_model 64) and the step's separate scan (above
    2048 lanes): containers of such weights are the oracle's, decode to the
    same bytes, and the steps' logits are the chunk forward's."""
    import torch

    import boa_hip
    w = tmp_path / "w.bin"
    _extreme_weights(w, d, 16)
    T = 9
    tok = np.random.default_rng(lanes).integers(0, 256, size=(lanes, T), dtype=np.uint8)
    c = boa_hip.Codec(d, 1, 16, lanes)
    c.set_stream(torch.cuda.current_stream().cuda_stream)
    c.load_weights(w)
    want = oracle.Model(w, d, 1, 16).new_state(lanes).forward_chunk(tok)
    c.reset_state(lanes)
    step = torch.zeros((lanes, 256), device="cuda")
    for t in range(T):
        c.step_batch(torch.from_numpy(tok[:, t].copy()).cuda(), lanes, step)
        torch.cuda.synchronize()
        assert np.array_equal(step.cpu().numpy().view(np.uint32), want[:, t].view(np.uint32))
    blob = c.compress(tok.tobytes(), chunk_size=T)
    assert blob == oracle.Model(w, d, 1).compress(tok.tobytes(), chunk_size=T)
    assert c.decompress(blob) == tok.tobytes()
    c.close()


def test_no_decay_matches_the_oracle(oracle, tmp_path):
    """A_log below -87: every decay coefficient is -0, the exponents are -0 and
    every ordinary token's scan runs without clamps."""
    import torch

    import boa_hip
    d, T = 64, 9
    w = tmp_path / "w.bin"
    synth.write_weights(str(w), [(name, np.full_like(a, -90.0) if name.endswith("A_log") else a)
                                 for name, a in synth.random_weight_tensors(d, 1, 16, seed=5)])
    lanes = 64 * 1024 // (2 * d)
    tok = np.random.default_rng(d).integers(0, 256, size=(lanes, T), dtype=np.uint8)
    want = oracle.Model(w, d, 1, 16).new_state(lanes).forward_chunk(tok)
    c = boa_hip.Codec(d, 1, 16, lanes)
    c.set_stream(torch.cuda.current_stream().cuda_stream)
    c.load_weights(w)
    c.reset_state(lanes)
    got = torch.zeros((lanes, T, 256), device="cuda")
    c.forward_chunk(torch.from_numpy(tok).cuda(), lanes, T, got)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy().view(np.uint32), want.view(np.uint32))
    c.close()
