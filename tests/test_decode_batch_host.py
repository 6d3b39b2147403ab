"""Which kernels a batched decode launches, on the host side of the library over a
stand-in for the HIP runtime: sequences of equal split counts a (splits, sequences)
grid, ragged ones one row of workgroups by the kernels made for it."""
import pytest

import hip_standin as hip
from hip_standin import PTR


@pytest.fixture(scope="module")
def ctx():
    with hip.binding().Context(0) as c:
        yield c


@pytest.mark.parametrize("Dh,lengths,kernel,grid", [
    (512, [4096] * 32, "g4a_decode_wave_batch_d512", (8, 32)),
    (256, [2048] * 16, "g4a_decode_wave_batch_d256", (16, 16)),
    (512, [8192, 4096, 512], "g4a_decode_wave_batch_row_d512", (200, 1)),
    (256, [8192, 4096, 512], "g4a_decode_wave_batch_row_d256", (200, 1)),
    (512, [320, 64], "g4a_decode_short_batch_row_d512", (12, 1)),
    (256, [320, 64], "g4a_decode_short_batch_d256", (10, 2)),
    (512, [320, 320], "g4a_decode_short_batch_d512", (10, 2)),
])
def test_grids(ctx, Dh, lengths, kernel, grid):
    calls = ctx.prepare_batch([dict(q=PTR, k=PTR, v=PTR, out=PTR, T=1, S=S, Hq=8, Hkv=1, Dh=Dh, Dv=Dh, q_pos0=S - 1)
                               for S in lengths])
    hip.launches()
    assert ctx.attention_decode_batch(calls) == len(lengths)
    first = hip.launches()[0]
    assert (first.name, first.gx, first.gy) == (kernel, *grid)
