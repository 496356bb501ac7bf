"""fp32 compress GEMM tiles: from 16,384 rows on the plain GEMMs of 256-wide
outputs run in 256-row persistent blocks, whose last tile starts early when
the rows are no multiple of 256, where those tiles pay.  The row counts here
are whole rounds of the CUs with 0, 1 and 255 rows over a tile, and 0.6 and 0.8
of a round.  The logits of every row equal those of calls of 4000 rows, whose
tiles are at most half of a round and so run on other kernels, and the rows
past the last one stay untouched."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,rows", [(64, 65281), (64, 65535), (256, 16384), (256, 65281),
                                    (256, 65535), (512, 65535), (64, 40001),
                                    (256, 40961)])
def test_rows_around_tiles(make_weights, d, rows):
    import torch

    import boa_hip
    c = boa_hip.Codec(d, 1, 16, rows)
    c.set_stream(torch.cuda.current_stream().cuda_stream)
    c.load_weights(make_weights(d, 1))
    tok = torch.from_numpy(np.random.default_rng(d).integers(0, 256, rows, dtype=np.uint8)).cuda()
    c.reset_state(rows)
    got = torch.full((rows + 300, 256), -7.0, device="cuda")
    c.forward_chunk(tok, rows, 1, got)
    want = torch.zeros((rows, 256), device="cuda")
    for r in range(0, rows, 4000):
        n = min(4000, rows - r)
        c.reset_state(n)
        c.forward_chunk(tok[r:r + n].contiguous(), n, 1, want[r:r + n])
    torch.cuda.synchronize()
    assert bool((got[rows:] == -7.0).all())
    assert torch.equal(got[:rows].view(torch.int32), want.view(torch.int32))
    c.close()


@pytest.mark.parametrize("d,rows", [(64, 15873), (80, 9001), (256, 3969), (256, 5505),
                                    (256, 16383), (512, 2049), (512, 8104)])
def test_mid_size_rows(make_weights, d, rows):
    """Fewer rows than a compress tile's run 128x64, 64x32 or 32x32 blocks by
    what they leave the fullest CU, or persistent blocks that fill the CUs: at
    rows around those lines the logits equal those of 200-row calls (32x32)."""
    import torch

    import boa_hip
    c = boa_hip.Codec(d, 1, 16, rows)
    c.set_stream(torch.cuda.current_stream().cuda_stream)
    c.load_weights(make_weights(d, 1))
    tok = torch.from_numpy(np.random.default_rng(rows).integers(0, 256, rows, dtype=np.uint8)).cuda()
    c.reset_state(rows)
    got = torch.full((rows + 300, 256), -7.0, device="cuda")
    c.forward_chunk(tok, rows, 1, got)
    want = torch.zeros((rows, 256), device="cuda")
    for r in range(0, rows, 200):
        n = min(200, rows - r)
        c.reset_state(n)
        c.forward_chunk(tok[r:r + n].contiguous(), n, 1, want[r:r + n])
    torch.cuda.synchronize()
    assert bool((got[rows:] == -7.0).all())
    assert torch.equal(got[:rows].view(torch.int32), want.view(torch.int32))
    c.close()
