"""Greedy hand-off over rows cut into parts: columns on both sides of a part's
edge, rows that start at every even address, strides other than N, short rows
and many rows (which one block walks), and tokens in pinned host memory, against
the first-maximum rule."""
import numpy as np
import pytest

from _ornith import from_dev
from oracle import ornith_oracle as O

pytestmark = pytest.mark.gpu

PART = 16384                       # columns per block


@pytest.mark.parametrize('M,N,lead', [(1, 1, 0), (2, 7, 3), (3, PART - 7, 7), (3, PART - 6, 7), (3, PART - 6, 1),
                                      (2, PART, 0), (2, PART + 1, 5), (5, 2 * PART + 9, 2), (1, 248320, 0),
                                      (33, 50001, 4), (3, 512, 1), (9, 513, 0), (9, 4096, 3), (9, 4097, 1),
                                      (520, 300, 5), (520, 2049, 6), (513, 2048, 1), (600, 519, 7), (512, 8192, 2),
                                      (512, 8193, 0), (2, 2 * PART, 1), (2, 2 * PART + 1, 1), (513, 3 * PART + 3, 4), (513, 1024, 1)])
@pytest.mark.parametrize('host', [False, True])
def test_argmax_parts(M, N, lead, host):
    import torch
    from ornith_g256 import native
    print(f'argmax M={M} N={N} lead={lead} host={host}', flush=True)
    rng = np.random.default_rng(N + lead)
    v = rng.standard_normal((M, N)).astype(np.float32)
    for r in range(M):             # the same maximum twice, at random and at part edges
        spots = [c for c in (N - 1, PART - lead, PART - lead - 1, 0, int(rng.integers(N))) if 0 <= c < N]
        v[r, rng.choice(spots, 2)] = 9.0
    if M > 2:
        v[1] = -np.inf             # all equal: column 0
        v[2, N - 1] = np.nan       # a late NaN beats every maximum
    bits = O.f32_to_bf16(v)
    pad = torch.full((M, N + lead + 3), float('inf'), dtype=torch.bfloat16, device='cuda')
    logits = pad[:, lead:lead + N]
    logits.copy_(torch.from_numpy(bits.view(np.int16)).cuda().view(torch.bfloat16))
    out = torch.full((M,), -1, dtype=torch.int64, pin_memory=True) if host else \
        torch.full((M,), -1, dtype=torch.int64, device='cuda')
    native.logits_argmax(logits, out)
    torch.cuda.synchronize()
    got = out.numpy() if host else from_dev(out)
    np.testing.assert_array_equal(got, O.argmax_first(O.bf16_to_f32(bits)))
