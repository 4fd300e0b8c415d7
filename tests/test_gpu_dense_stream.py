"""Weight-streaming dense linears at the edges of their row tiles (4, 8, 16, 32
and 64 rows), of a block's waves (4, 8 and 16 groups of K, and one more) and of
its 32 columns, bit for bit against the oracle."""
import numpy as np
import pytest

from _ornith import Bank, bf16_normal, from_dev, to_dev
from oracle import ornith_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('M,N,K,tile', [(4, 48, 1280, 16), (5, 64, 1024, 32), (8, 16, 1024, 16), (9, 80, 1280, 16),
                                        (16, 32, 2304, 32), (17, 48, 4096, 16), (32, 96, 2048, 16),
                                        (32, 16, 4352, 16), (33, 48, 2048, 16), (49, 32, 512, 16), (64, 80, 2304, 16)])
def test_dense_stream_edges(M, N, K, tile):
    import torch
    from ornith_g256 import native
    print(f'dense stream M={M} N={N} K={K} tile={tile}', flush=True)
    rng = np.random.default_rng(M * 31 + N + K)
    bank = Bank(rng, 0, N, K, tile=tile)
    x = bf16_normal(rng, (M, K))
    x[M // 2] = 0                              # an all-zero row
    ref_out, _, ref_flags = O.dense_a8(x, *bank.expert())
    ws = torch.empty(native.dense_layout(64, N, K).workspace_bytes, dtype=torch.uint8, device='cuda')
    out = torch.full((M + 1, N), -1.0, dtype=torch.bfloat16, device='cuda')
    flags = torch.zeros(1, dtype=torch.int32, device='cuda')
    xd, cd, md = (to_dev(v, torch.device('cuda')) for v in (x, bank.codes, bank.meta))
    h = native.lib()
    fn = h.ornith_dense_g256_launch if tile == 16 else h.ornith_dense_g256_launch_n32
    assert fn(native.ptr(xd), native.ptr(cd), native.ptr(md), native.ptr(ws), ws.numel(), native.ptr(out),
              native.ptr(flags), M, 64, N, K, 8, 128, 2, native.stream(xd)) == 0
    torch.cuda.synchronize()
    np.testing.assert_array_equal(from_dev(out[:M].contiguous()), ref_out)
    assert (out[M] == -1).all()                # rows past M are left alone
    assert int(flags.item()) == ref_flags
