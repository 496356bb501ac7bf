"""bf16 compress GEMM tiles: row counts around the 256-row tiles and their
spread over the eight XCDs (one tile, whole tiles, one row over, more blocks
than an XCD's share), at every built bf16 width (K from 64 to 2048, 256- to
2048-feature outputs).  The decode step runs other kernels with the same
MFMA chains, so its logits have to be the chunk forward's bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,ds", [(64, 16), (128, 16), (256, 16), (512, 32)])
@pytest.mark.parametrize("lanes,T", [(1, 1), (85, 3), (128, 2), (257, 1), (683, 3)])
def test_rows_around_tiles(make_weights, d, ds, lanes, T):
    import torch

    import boa_hip
    c = boa_hip.Codec(d, 2, ds, lanes, precision="bf16")
    c.set_stream(torch.cuda.current_stream().cuda_stream)
    c.load_weights(make_weights(d, 2, ds))
    tok = np.random.default_rng(lanes + d).integers(0, 256, size=(lanes, T), dtype=np.uint8)
    c.reset_state(lanes)
    # rows past the last one must stay as they are
    out = torch.full((lanes * T + 300, 256), -7.0, device="cuda")
    c.forward_chunk(torch.from_numpy(tok).cuda(), lanes, T, out)
    torch.cuda.synchronize()
    assert bool((out[lanes * T:] == -7.0).all())
    got = out[:lanes * T].cpu().numpy().reshape(lanes, T, 256)
    c.reset_state(lanes)
    step = torch.zeros((lanes, 256), device="cuda")
    for t in range(T):
        c.step_batch(torch.from_numpy(tok[:, t].copy()).cuda(), lanes, step)
        torch.cuda.synchronize()
        assert np.array_equal(step.cpu().numpy().view(np.uint32), got[:, t].copy().view(np.uint32))
    c.close()


@pytest.mark.parametrize("layers", [1, 3])
@pytest.mark.parametrize("rows", [32768, 32769, 32897, 33151, 65535])
def test_feed_forward_by_rows(make_weights, layers, rows):
    """d_model 256: from 257 blocks of 128 rows on the feed-forward pair runs
    by rows (with LN2, and LN1 where a layer follows).  Around that line, with
    1, 127 and 128 rows in the last block, the logits equal those of short
    calls, and the rows past the last one stay untouched."""
    import torch

    import boa_hip
    c = boa_hip.Codec(256, layers, 16, rows, precision="bf16")
    c.set_stream(torch.cuda.current_stream().cuda_stream)
    c.load_weights(make_weights(256, layers))
    tok = torch.from_numpy(np.random.default_rng(rows).integers(0, 256, rows, dtype=np.uint8)).cuda()
    c.reset_state(rows)
    got = torch.full((rows + 300, 256), -7.0, device="cuda")
    c.forward_chunk(tok, rows, 1, got)
    want = torch.zeros((rows, 256), device="cuda")
    for r in range(0, rows, 8192):
        n = min(8192, rows - r)
        c.reset_state(n)
        c.forward_chunk(tok[r:r + n].contiguous(), n, 1, want[r:r + n])
    torch.cuda.synchronize()
    assert bool((got[rows:] == -7.0).all())
    assert torch.equal(got[:rows].view(torch.int32), want.view(torch.int32))
    c.close()
