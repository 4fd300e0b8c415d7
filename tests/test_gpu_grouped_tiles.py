"""Layers of more than 32 tokens (grouped projections in 16- and 32-route
m-tiles) against the same tokens in batches of 24, which take the decode
kernels: bit for bit, at the edges of the tiles, of the tile rules (64, 192,
512, 576, 1024, 2048 and 5120 tokens) and with experts of 1 to several tiles' routes."""
import numpy as np
import pytest

from _ornith import Bank, bf16_normal, from_dev, load_shared_tables, moe_weights, random_routing, to_dev

pytestmark = pytest.mark.gpu
DISTINCT = 24
SIZES = [33, 47, 64, 65, 129, 192, 193, 300, 512, 513, 577, 1024, 1120, 2048, 2049, 5120, 5121]


def _tokens(rng, T):
    """T tokens out of DISTINCT, skewed, so that counts per expert spread."""
    return np.minimum(rng.geometric(0.2, size=T) - 1, DISTINCT - 1).astype(np.int64)


@pytest.fixture(scope='module')
def banks():
    import torch
    dev = torch.device('cuda')
    rng = np.random.default_rng(77)
    raw = {tile: (Bank(rng, 256, 1024, 2048, tile=tile), Bank(rng, 256, 2048, 512, tile=tile)) for tile in (16, 32)}
    return {t: [v for b in pair for v in (to_dev(b.codes, dev), to_dev(b.meta, dev))] for t, pair in raw.items()}


def _routed(native, tile, entry, bank, x, w, ids):
    import torch
    T = x.shape[0]
    ws = torch.empty(native.routed_layout(T, tile=tile).workspace_bytes, dtype=torch.uint8, device='cuda')
    out = torch.full((T + 1, 2048), -1.0, dtype=torch.bfloat16, device='cuda')
    flags = torch.zeros(1, dtype=torch.int32, device='cuda')
    args = [native.ptr(t) for t in (x, w, ids, *bank, ws)]
    assert getattr(native.lib(tile), entry)(*args, ws.numel(), native.ptr(out), native.ptr(flags), T, T,
                                            native.stream(x)) == 0
    torch.cuda.synchronize()
    assert (out[T] == -1).all()                # rows past T are left alone
    return out[:T], int(flags.item())


@pytest.mark.parametrize('tile,entry', [(32, 'ornith_routed_direct_launch'), (16, 'ornith_routed_direct_launch'),
                                        (16, 'ornith_routed_direct_launch_a4')])
@pytest.mark.parametrize('T', SIZES)
def test_routed_matches_small_batches(banks, T, tile, entry):
    import torch
    from ornith_g256 import native
    print(f'routed T={T} tile={tile} {entry}', flush=True)
    dev = torch.device('cuda')
    rng = np.random.default_rng(T)
    x = bf16_normal(rng, (DISTINCT, 2048))
    x[3] = 0                                   # an all-zero row
    x[5, 100] = 0x7F80                         # a non-finite one
    w, ids = random_routing(rng, DISTINCT)
    ids[:, 0] = 9                              # one expert for every token
    ids[7, 2:5] = -1                           # dead slots
    ids[8, 1] = 300                            # an invalid expert
    pick = _tokens(rng, T)
    pick[:DISTINCT] = np.arange(DISTINCT)
    bank = list(banks[tile])
    if entry.endswith('a4'):                   # metadata that starts at an odd word
        for k in (1, 3):
            bank[k] = torch.cat([bank[k].flatten()[:1], bank[k].flatten()])[1:]
            assert bank[k].data_ptr() % 8 == 4
    ref, ref_flags = _routed(native, tile, entry, banks[tile], *(to_dev(v, dev) for v in (x, w, ids)))
    got, flags = _routed(native, tile, entry, bank, *(to_dev(v[pick], dev) for v in (x, w, ids)))
    np.testing.assert_array_equal(from_dev(got), from_dev(ref)[pick])
    assert flags == ref_flags and flags & 5 == 5


@pytest.fixture(scope='module')
def layer():
    import torch
    dev = torch.device('cuda')
    w = moe_weights(4321)
    d = {k: (to_dev(v.codes, dev), to_dev(v.meta, dev)) for k, v in w.items() if isinstance(v, Bank)}
    router, gate = to_dev(w['router'], dev), to_dev(w['gate'][0], dev)
    silu, sigmoid = (to_dev(t, dev) for t in load_shared_tables())
    return d, router, gate, silu, sigmoid


@pytest.mark.parametrize('T', SIZES)
def test_layer_matches_small_batches(layer, T):
    import torch
    from ornith_g256 import native
    print(f'layer T={T}', flush=True)
    dev = torch.device('cuda')
    d, router, gate, silu, sigmoid = layer
    rng = np.random.default_rng(T)
    x = bf16_normal(rng, (DISTINCT, 2048))
    pick = _tokens(rng, T)

    def run(rows):
        n = rows.shape[0]
        ws = torch.zeros(native.routed_layout(n, 'layer').workspace_bytes, dtype=torch.uint8, device=dev)
        out = torch.empty((n, 2048), dtype=torch.bfloat16, device=dev)
        tw = torch.empty((n, 8), dtype=torch.float32, device=dev)
        ti = torch.empty((n, 8), dtype=torch.int32, device=dev)
        sl = torch.empty((n,), dtype=torch.bfloat16, device=dev)
        flags = torch.zeros(1, dtype=torch.int32, device=dev)
        native.moe_layer(to_dev(rows, dev), router, None, gate, *d['w13'], *d['w2'], *d['s13'], *d['s2'], silu,
                         sigmoid, ws, tw, ti, sl, out, flags, n)
        torch.cuda.synchronize()
        assert int(flags.item()) == 0
        return from_dev(out), from_dev(ti)
    ref, ref_ids = run(x)
    got, ids = run(x[pick])
    np.testing.assert_array_equal(ids, ref_ids[pick])
    np.testing.assert_array_equal(got, ref[pick])
