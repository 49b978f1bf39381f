"""The index math of the set_points kernels (mripy_amd/csrc/gn_kernels.hip), restated in NumPy
with a bounds assertion on every index, no GPU needed:

* k_scan / k_pair_scan / k_item_scan: tiles scanned in place, block totals turned into
  offsets by the last block, consumers adding data[i] + bsum[i / tile];
* k_radix_count / k_radix_scatter: one count per workgroup's chunk, the scatter's four
  quarters counted again, run starts in wave order, 64 items a step;
* k_pair_keys / k_pair_records: pairs at the tiled offsets, their tiles decoded from the
  sorted key;
* k_item_write for spread and gather items at every item length, and the buffers' sizes.
"""
import numpy as np
import pytest

from test_setpoints_emulation import axis_tile_span, axis_tiles, default_tiles, prep, spread_items_host, tap_box

SCAN_THREADS, SCAN_ITEMS = 256, 8
SCAN_TILE = SCAN_THREADS * SCAN_ITEMS
ITEM_TILE = SCAN_THREADS * 4
RADIX_BITS, WAVES, UNROLL = 11, 4, 4
GATHER_CHUNK = 512


def scan(x, capacity, tile=SCAN_TILE):
    """(data, bsum): exclusive scan within tiles, block offsets and the grand total last."""
    n = x.shape[0]
    nb = max(1, -(-n // tile))
    assert nb + 1 <= capacity
    data = np.zeros_like(x)
    totals = np.zeros((nb,) + x.shape[1:], np.int64)
    for b in range(nb):
        v = x[b * tile:(b + 1) * tile]
        data[b * tile:(b + 1) * tile] = np.cumsum(v, 0) - v
        totals[b] = v.sum(0)
    # the last block: 256 totals at a time behind a carry
    bsum = np.zeros((nb + 1,) + x.shape[1:], np.int64)
    carry = np.zeros(x.shape[1:], np.int64)
    for b0 in range(0, nb, SCAN_THREADS):
        v = totals[b0:b0 + SCAN_THREADS]
        bsum[b0:b0 + v.shape[0]] = np.cumsum(v, 0) - v + carry
        carry = carry + v.sum(0)
    bsum[nb] = carry
    return data, bsum


def digit_pass(keys, vals, shift, bits, chunk_len):
    n = keys.shape[0]
    bins = 1 << bits
    C = max(1, -(-n // chunk_len))
    digit = (keys >> shift) & (bins - 1)
    cnt = np.full(bins * C, -1, np.int64)
    for c in range(C):
        cnt[np.arange(bins) * C + c] = np.bincount(digit[c * chunk_len:min(n, (c + 1) * chunk_len)], minlength=bins)
    assert (cnt >= 0).all()
    offs, bsum = scan(cnt, bins * C // SCAN_TILE + 2)
    kout, vout = np.full(n, -1, np.int64), np.full(n, -1, np.int64)
    part = chunk_len // WAVES
    assert part * WAVES == chunk_len and part % 64 == 0
    for c in range(C):
        quarters = [(min(n, c * chunk_len + w * part), min(n, c * chunk_len + (w + 1) * part)) for w in range(WAVES)]
        i = np.arange(bins) * C + c
        run = offs[i] + bsum[i // SCAN_TILE]
        base = []
        for b, e in quarters:
            base.append(run.copy())
            run = run + np.bincount(digit[b:e], minlength=bins)
        for w, (b, e) in enumerate(quarters):
            for g in range(b, e, 64):
                d = digit[g:min(e, g + 64)]
                eq = d[:, None] == d[None, :]
                rank = np.tril(eq, -1).sum(1)
                at = base[w][d] + rank
                assert (at >= 0).all() and (at < n).all() and (kout[at] == -1).all()
                kout[at], vout[at] = keys[g:g + d.size], vals[g:g + d.size]
                np.add.at(base[w], d, 1)
    return kout, vout


def stable_sort(keys, vals, K):
    kbits = 1
    while kbits < 31 and (1 << kbits) < K:
        kbits += 1
    npass = -(-kbits // RADIX_BITS)
    pbits = -(-kbits // npass)
    n = keys.shape[0]
    wave = min(4096, max(256, -(-(-(-n // 4096)) // 64) * 64))
    shift = 0
    for _ in range(npass):
        bits = min(pbits, kbits - shift)
        keys, vals = digit_pass(keys, vals, shift, bits, WAVES * wave)
        shift += bits
    assert shift == kbits
    return keys, vals


def bin_starts(skeys, K):
    n = skeys.shape[0]
    out = np.full(K + 1, -1, np.int64)
    for i in range(n + 1):
        prev = -1 if i == 0 else skeys[i - 1]
        nxt = K if i == n else skeys[i]
        out[prev + 1:nxt + 1] = i
    assert (out >= 0).all()
    return out


def device_items(start, chunk, spread):
    """k_item_scan and k_item_write; capacities as bin_and_sort allocates them."""
    K = start.shape[0] - 1
    n = np.diff(start)
    nch = -(-n // chunk)
    counts = np.stack([nch, n == 0, np.where(n > chunk, nch, 0), n > chunk], 1).astype(np.int64)
    off, bsum = scan(counts, -(-K // ITEM_TILE) + 1, ITEM_TILE)
    P = int(start[-1])
    cap = K + P // chunk + 1
    items, red = [None] * cap, [None] * max(1, min(K, P // chunk + 1))
    for k in range(K):
        o, s = off[k], bsum[k // ITEM_TILE]
        b, e = int(start[k]), int(start[k + 1])
        if e == b:
            if spread:
                i = int(bsum[-1][0] + o[1] + s[1])
                assert items[i] is None
                items[i] = (k, b, e, -1)
            continue
        i0 = int(o[0] + s[0])
        if spread and e - b <= chunk:
            assert items[i0] is None
            items[i0] = (k, b, e, -1)
            continue
        s0 = int(o[2] + s[2])
        for c, x in enumerate(range(b, e, chunk)):
            assert items[i0 + c] is None
            items[i0 + c] = (k, x, min(e, x + chunk), s0 + c if spread else 0)
        if spread:
            r = int(o[3] + s[3])
            assert red[r] is None
            red[r] = (k, s0, -(-(e - b) // chunk), 0)
    full, empty, slots, nred = (int(v) for v in bsum[-1])
    return items[:full + (empty if spread else 0)], red[:nred], slots


@pytest.mark.parametrize("n", [1, 2047, 2048, 2049, SCAN_TILE * 300 + 5])
def test_tiled_scan(n):
    x = np.random.default_rng(n).integers(0, 9, n)
    data, bsum = scan(x, n // SCAN_TILE + 2)
    i = np.arange(n)
    assert np.array_equal(data + bsum[i // SCAN_TILE], np.cumsum(x) - x) and bsum[-1] == x.sum()


@pytest.mark.parametrize("n,K", [(1, 1), (63, 2), (1024, 300), (1025, 5000), (5000, 1 << 17), (4096 * 256 + 70, 40000)])
def test_sort_by_workgroup_chunks(n, K):
    rng = np.random.default_rng(n)
    keys = np.where(rng.random(n) < 0.4, rng.integers(0, max(1, K // 20), n), rng.integers(0, K, n))
    vals = rng.permutation(n)
    k, v = stable_sort(keys, vals, K)
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(k, keys[order]) and np.array_equal(v, vals[order])


@pytest.mark.parametrize("modes,ns,rat,M,tiles", [((16, 20, 18), 3, 2, 1500, None), ((12, 9, 10), 5, 2, 400, None),
                                                  ((5, 4, 6), 8, 2, 60, None), ((6, 6, 6), 3, 2, 200, (1, 1, 1)),
                                                  ((64, 50), 3, 2, 2500, None), ((7, 9), 3, 2, 300, None),
                                                  ((16, 16), 14, 3, 500, None), ((20, 22), 4, 2, 300, (3, 5))])
@pytest.mark.parametrize("cluster", [False, True])
def test_pairs_and_items(modes, ns, rat, M, tiles, cluster):
    rng = np.random.default_rng(sum(modes) + ns)
    dim, W = len(modes), 2 * ns
    nf = [max(rat * m, W) for m in modes]
    tile, gtile = default_tiles(dim, ns, nf)
    if tiles:
        tile = [t if t + W - 1 <= n else d for t, n, d in zip(tiles, nf, tile)]
    coords = [np.pi * (2 * rng.random(M) - 1) if not cluster else 0.05 * rng.standard_normal(M) for _ in modes]
    s, _, key, ng = prep(coords, nf, ns, gtile)
    Kg = int(np.prod(ng))
    skeys, order = stable_sort(key, np.arange(M), Kg)
    assert np.array_equal(order, np.argsort(key, kind="stable"))
    start = bin_starts(skeys, Kg)
    cells = np.stack([a[order] for a in s], 1)
    # k_pair_scan, k_pair_keys
    ntiles = [-(-nf[a] // tile[a]) for a in range(dim)]
    K = int(np.prod(ntiles))
    spans = [[axis_tile_span(int(c[a]), W, nf[a], tile[a]) for a in range(dim)] for c in cells]
    cnt = np.array([int(np.prod([n for _, n in sp])) for sp in spans])
    offs, bsum = scan(cnt, -(-M // SCAN_TILE) + 1)
    P = int(bsum[-1])
    pkey, psamp = np.full(P, -1), np.full(P, -1)
    for p, sp in enumerate(spans):
        o = int(offs[p] + bsum[p // SCAN_TILE])
        for local in np.ndindex(*[n for _, n in sp]):
            k = 0
            for a in range(dim):
                t = sp[a][0] + local[a]
                t -= ntiles[a] if t >= ntiles[a] else 0
                assert 0 <= t < ntiles[a]
                k = k * ntiles[a] + t
            assert 0 <= o < P and pkey[o] == -1
            pkey[o], psamp[o] = k, p
            o += 1
    assert (pkey >= 0).all()
    # sort carrying the samples; k_pair_records decodes the tile from the key
    sk, samp = stable_sort(pkey, psamp, K)
    ref = np.argsort(pkey, kind="stable")
    assert np.array_equal(samp, psamp[ref])
    pstart = bin_starts(sk, K)
    assert pstart[-1] == P
    for q in range(P):
        k, p = int(sk[q]), int(samp[q])
        t = []
        for a in reversed(range(dim)):
            t.append(k % ntiles[a])
            k //= ntiles[a]
        assert k == 0
        for a, qt in enumerate(reversed(t)):
            assert qt in axis_tiles(int(cells[p, a]), W, nf[a], tile[a])
            j, c, l0 = tap_box(int(cells[p, a]), qt, tile[a], nf[a], W)
            assert 0 <= j < 256 and 1 <= c < 256 and 0 <= l0 < 1024 and j + c <= W
            assert tile[a] == nf[a] or l0 + c <= min(tile[a], nf[a] - qt * tile[a])
    for chunk in (128, 192, 256, 448, 512):
        assert device_items(pstart, chunk, True) == spread_items_host(pstart, chunk)
    gather, _, _ = device_items(start, GATHER_CHUNK, False)
    assert gather == [(k, x, min(int(start[k + 1]), x + GATHER_CHUNK), 0) for k in range(Kg)
                      for x in range(int(start[k]), int(start[k + 1]), GATHER_CHUNK)]


@pytest.mark.parametrize("nt0,ncolt", [(1, 5), (63, 3), (64, 4), (65, 2), (200, 7)])
def test_occupancy_words(nt0, ncolt):
    """k_occ_masks: a lane per group of mask_k leading-axis tiles, waves looping over columns."""
    rng = np.random.default_rng(nt0)
    cnt = (rng.random(nt0 * ncolt) < 0.3).astype(np.int64) * rng.integers(1, 9, nt0 * ncolt)
    pstart = np.concatenate([[0], np.cumsum(cnt)])
    mask_k = -(-nt0 // 64)
    blocks = 1 if ncolt > 4 else 2
    got = np.zeros(ncolt, object)
    seen = np.zeros(ncolt, int)
    for b in range(blocks):
        for w in range(4):
            for c in range(b * 4 + w, ncolt, blocks * 4):
                m = 0
                for lane in range(64):
                    for t0 in range(lane * mask_k, min(nt0, (lane + 1) * mask_k)):
                        k = t0 * ncolt + c
                        assert 0 <= k and k + 1 < pstart.size
                        if pstart[k + 1] > pstart[k]:
                            m |= 1 << lane
                got[c] = m
                seen[c] += 1
    assert (seen == 1).all()
    for c in range(ncolt):
        assert got[c] == sum(1 << g for g in range(64) if any(cnt[t * ncolt + c] for t in range(g * mask_k, min(nt0, (g + 1) * mask_k))))
