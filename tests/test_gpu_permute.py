"""The permutation, read back from the workspace after a layer call.

The prefill path (T > 32) sorts the routes into banks
(routed_storage_n32_prefill.h:19-42 computes the same counts, offsets and
per-expert route lists; its list order is atomic, this library's is stable).
Here what the kernels wrote is compared with the oracle's ``permute``
on the ids the kernels themselves produced (the layer entry's router + top-8,
and the routed entry's caller ids with duplicates and invalid entries):

  * per 16-token block and bank, the block's count (up to 2048 tokens, where
    each scatter block sums them itself) or the running count over the earlier
    blocks (the scan's output), and then the bank totals;
  * the permuted route list: ascending route index within each bank, the
    shared routes R + t after the routed ones;
  * the m-tiles the projections read, {bank, first route, rows, tile in bank} of
    the non-empty banks (bank 256 = shared expert), and their number, at the
    tile heights of both bank widths.

The workspace offsets follow the library's workspace plan: the m-tiles start at
``gate_y``, the permutation scratch at the first 256-byte boundary after
``final_f32`` (T x 2048 fp32), carved into 256-byte aligned arrays.
"""
import numpy as np
import pytest

from _ornith import bf16_normal, from_dev, moe_weights, random_routing, to_dev
from oracle import ornith_oracle as O

pytestmark = pytest.mark.gpu

E, BANKS, TOP, PERM_TOKENS, FUSED_TOKENS = 256, 257, 8, 16, 2048


def _tile_rows(T, bank_tile):
    """Routes per m-tile of a layer of T tokens (the projections' rule)."""
    if bank_tile == 32:
        return 16 if T <= 512 else 32
    return 16 if T <= 192 or 576 < T <= 1024 else 32


def _a256(n):
    return (n + 255) & ~255


def _carve(ws, layout, Tcap, shared):
    """Views of the m-tiles and the permutation scratch inside the workspace bytes."""
    rall = Tcap * (TOP + (1 if shared else 0))
    blocks = (Tcap + PERM_TOKENS - 1) // PERM_TOKENS
    out, off = {'tiles': ws[layout.gate_y:layout.middle].view(np.int32)}, _a256(layout.final_f32 + Tcap * 2048 * 4)
    for name, n in [('block_counts', blocks * E), ('counts', E), ('routes', rall), ('ntiles', 1)]:
        out[name] = ws[off:off + 4 * n].view(np.int32)
        off += _a256(4 * n)
    return out


def _expected(ids, T, shared, rows):
    R = T * TOP
    ids = np.asarray(ids, np.int32).reshape(-1)
    counts, offsets, routes = O.permute(ids)
    s = T if shared else 0
    counts = np.append(counts, s).astype(np.int32)
    offsets = np.append(offsets, offsets[-1] + s).astype(np.int32)
    routes = np.concatenate([routes, R + np.arange(s, dtype=np.int32)])
    tiles = [(b, offsets[b] + k, min(rows, counts[b] - k), k // rows)
             for b in range(BANKS) for k in range(0, counts[b], rows)]
    nblocks = (T + PERM_TOKENS - 1) // PERM_TOKENS
    valid = (ids >= 0) & (ids < E)
    per_block = np.zeros((nblocks, E), np.int64)
    np.add.at(per_block, (np.arange(R)[valid] // (PERM_TOKENS * TOP), ids[valid]), 1)
    return counts, routes, np.array(tiles, np.int32).reshape(-1, 4), per_block


def _check(p, ids, T, shared, rows):
    counts, routes, tiles, per_block = _expected(ids, T, shared, rows)
    np.testing.assert_array_equal(p['routes'][:len(routes)], routes)
    assert int(p['ntiles'][0]) == len(tiles)
    np.testing.assert_array_equal(p['tiles'][:4 * len(tiles)].reshape(-1, 4), tiles)
    left = per_block
    if T > FUSED_TOKENS:
        left = np.cumsum(per_block, axis=0) - per_block
        np.testing.assert_array_equal(p['counts'], counts[:E])
    np.testing.assert_array_equal(p['block_counts'].reshape(-1, E)[:len(left)], left)
    return counts


def _zipf_bias(s, seed):
    rank = np.random.default_rng(seed).permutation(256).astype(np.float64) + 1.0
    return (-s * np.log(rank)).astype(np.float32)


@pytest.fixture(scope='module')
def banks(device):
    w = moe_weights(1234)
    d = {k: (to_dev(w[k].codes, device), to_dev(w[k].meta, device)) for k in ('w13', 'w2', 's13', 's2')}
    return w, d


@pytest.mark.parametrize('tile', [32, 16])
@pytest.mark.parametrize('T,zipf', [(33, None), (192, None), (193, None), (300, None), (300, 1.3), (513, 1.1),
                                    (577, None), (1024, 1.1), (1025, None), (1120, 1.1), (2048, 1.3), (2049, 1.3),
                                    (5121, None)])
def test_layer_permutation_matches_oracle(device, banks, shared_tables, T, zipf, tile):
    import torch
    from ornith_g256 import native
    w, d = banks
    silu, sigmoid = shared_tables
    print(f'permutation: layer T={T} zipf={zipf} tile={tile}', flush=True)
    rng = np.random.default_rng(9100 + T)
    x = to_dev(bf16_normal(rng, (T, 2048)), device)
    bias = None if zipf is None else to_dev(_zipf_bias(zipf, 11), device)
    layout = native.routed_layout(T, 'layer', tile)
    ws = torch.full((layout.workspace_bytes,), 0xA5, dtype=torch.uint8, device=device)   # no stale zeros
    out = torch.empty((T, 2048), dtype=torch.bfloat16, device=device)
    tw = torch.empty((T, 8), dtype=torch.float32, device=device)
    ti = torch.empty((T, 8), dtype=torch.int32, device=device)
    sl = torch.empty((T,), dtype=torch.bfloat16, device=device)
    flags = torch.zeros(1, dtype=torch.int32, device=device)
    native.moe_layer(x, to_dev(w['router'], device), bias, to_dev(w['gate'][0], device),
                     d['w13'][0], d['w13'][1], d['w2'][0], d['w2'][1], d['s13'][0], d['s13'][1],
                     d['s2'][0], d['s2'][1], to_dev(silu, device), to_dev(sigmoid, device),
                     ws, tw, ti, sl, out, flags, T, tile)
    torch.cuda.synchronize()
    assert int(flags.item()) == 0
    ids = from_dev(ti)
    rows = _tile_rows(T, tile)
    counts = _check(_carve(from_dev(ws), layout, T, True), ids, T, True, rows)
    if zipf is not None:
        assert counts[:E].max() > rows           # a bank with several m-tiles
    print(f'  banks used {int((counts[:E] > 0).sum())}, top bank {int(counts[:E].max())} routes', flush=True)


def test_routed_entry_permutation_with_edge_ids(device, banks):
    """Caller ids: duplicates within a token, padding (-1) and out-of-range
    ids (skipped and flagged), one bank in several m-tiles."""
    import torch
    from ornith_g256 import native
    w, d = banks
    T = 70
    print(f'permutation: routed entry T={T} edge ids', flush=True)
    rng = np.random.default_rng(9177)
    x = to_dev(bf16_normal(rng, (T, 2048)), device)
    rw, ids = random_routing(rng, T)
    ids[ids == 3] = 4                                  # bank 3 only in slot 0: five m-tiles
    ids[:, 0] = 3
    ids[2, :] = 9                                      # a token naming one expert eight times
    ids[4, 5] = -1                                     # padding
    ids[6, 2] = 300                                    # invalid: skipped, flag 4
    ids[8, 7] = -2                                     # invalid: skipped, flag 4
    layout = native.routed_layout(T)
    ws = torch.full((layout.workspace_bytes,), 0x5A, dtype=torch.uint8, device=device)
    out = torch.empty((T, 2048), dtype=torch.bfloat16, device=device)
    flags = torch.zeros(1, dtype=torch.int32, device=device)
    st = native.lib().ornith_routed_direct_launch(
        *[native.ptr(t) for t in (x, to_dev(rw, device), to_dev(ids, device), d['w13'][0], d['w13'][1],
                                  d['w2'][0], d['w2'][1], ws)],
        ws.numel(), native.ptr(out), native.ptr(flags), T, T, native.stream(x))
    assert st == 0
    torch.cuda.synchronize()
    assert int(flags.item()) & 4
    counts = _check(_carve(from_dev(ws), layout, T, False), ids, T, False, _tile_rows(T, 32))
    assert counts[3] > 64 and counts[9] >= 8
