"""Synthetic cohorts for the message kernels: random suffix words, keys, routing tags in every combination the kernels
branch on (suffix below ctx, below ctx / 2, retired recipients, pill receipts, retiring senders)."""
import numpy as np


def cohort(n, p, ctx, packed, seed):
    rng = np.random.default_rng(seed)
    suf = rng.integers(0, 4 * ctx + 1000, n).astype(np.uint64)
    suf[: min(n, 8)] = np.array([0, ctx - 1, ctx, ctx // 2, max(ctx // 2 - 1, 0), ctx + 1, 3 * ctx, 1], dtype=np.uint64)[: min(n, 8)]
    tag = rng.integers(0, 1 << 16, n).astype(np.uint64)
    sa = suf | (tag << np.uint64(48))                       # the forward tag rides in the top 16 bits of a word
    cur = rng.integers(0, p, n).astype(np.uint32) | (np.uint32(0x8000) * (rng.random(n) < 0.2))
    prev = rng.integers(0, p, n).astype(np.uint32) | (np.uint32(0x8000) * (rng.random(n) < 0.2))
    beta = (prev.astype(np.uint32) << np.uint32(16)) | cur.astype(np.uint32)
    if packed:
        primary = rng.integers(0, 1 << 31, n).astype(np.uint64)
        secondary = rng.integers(0, 1 << 31, n).astype(np.uint64)
        pill = (rng.random(n) < 0.3).astype(np.uint64)
        keys = (primary << np.uint64(31)) | secondary | (pill << np.uint64(62))
    else:
        keys = rng.integers(0, 1 << 31, n).astype(np.uint64)
    active_sz = int(rng.integers(0, n + 1))
    return sa, keys, beta.astype(np.uint32), active_sz


def groups(target, rank, end, p):
    """The messages of every destination as a sorted list, whatever their order inside the group."""
    start = 0
    out = []
    for q in range(p):
        e = int(end[q])
        out.append(sorted(zip(target[start:e].tolist(), rank[start:e].tolist())))
        start = e
    return out


def runs_of_first_words(key_words, long_runs, seed):
    """Keys of generation 0 with runs of one first word as long as a tile sorts in place (256), one shorter and one longer, and across
    the ends of tiles of 1024; the other words and the forward tags differ, or only the last of them does, or nothing does. long_runs: "few", of a list that goes on with
    short ones, or "many", when runs of up to 32 are sorted in place, with some on both sides of that."""
    rng = np.random.default_rng(seed)
    lengths = [1, 2, 255, 256, 3, 1, 500 - (1 + 2 + 255 + 256 + 3 + 1) % 500, 256, 255, 2, 17] + rng.integers(1, 6, 900).tolist()
    if long_runs == "few":
        lengths += [257, 300, 2] + rng.integers(1, 6, 6000).tolist()
    elif long_runs == "many":
        lengths += [31, 32, 33, 34, 1] * 5 + [900, 64, 128] * 6
    elif long_runs:
        lengths += [257, 1, 700, 2500, 2, 256]
    first = np.repeat(np.cumsum(rng.integers(1, 1 << 40, len(lengths))).astype(np.uint64), lengths)
    if not long_runs:  # (one of the lengths above is longer than a tile sorts)
        first[518:1000] += np.arange(482, dtype=np.uint64) // np.uint64(2)
    m = first.size
    keys = np.zeros((m, key_words), dtype=np.uint64)
    keys[:, 0] = first
    for w in range(1, key_words):
        keys[:, w] = rng.integers(0, 3, m).astype(np.uint64) << np.uint64(62)  # (the words are unsigned)
    tags = rng.integers(0, 2, m).astype(np.uint32) * np.uint32(40000)
    lanes = rng.permutation(m).astype(np.uint64) + np.uint64(1 << 33)
    order = rng.permutation(m)
    return keys[order], lanes[order], tags[order] << np.uint32(16)


def check_runs_of_first_words(lib, to_dev, to_host, handle, key_words, long_runs):
    """csa_sort_init_dev of one partition against a sort by (words, forward tag, place): ranks, lanes and the active set."""
    import ctypes as C
    import oracle_lib
    from cascade_amd import _native
    keys, lanes, beta = runs_of_first_words(key_words, long_runs, 7 * key_words)
    m = lanes.size
    d_keys, d_lanes, d_beta = to_dev(keys.reshape(-1)), to_dev(oracle_lib.u64_to_sa40(lanes)), to_dev(beta)
    d_rank, d_suf = to_dev(np.zeros(m, dtype=np.uint32)), to_dev(np.zeros(5 * m, dtype=np.uint8))
    d_mt, d_mr, d_off = to_dev(np.zeros(10 * m, dtype=np.uint8)), to_dev(np.zeros(2 * m, dtype=np.uint32)), to_dev(np.zeros(2, dtype=np.uint32))
    res = _native.CsaStepResult()
    h = handle(m)
    try:
        assert lib.csa_sort_init_dev(h, d_keys.ptr, key_words, d_lanes.ptr, d_beta.ptr, m, 1, d_rank.ptr, d_suf.ptr, d_mt.ptr, d_mr.ptr,
                                     d_off.ptr, None, C.byref(res)) == 0, lib.csa_last_error()
        got_rank, got_suf = to_host(d_rank), oracle_lib.sa40_to_u64(to_host(d_suf))
    finally:
        lib.csa_destroy(h)
    columns = [beta >> np.uint32(16)] + [keys[:, w] for w in reversed(range(key_words))]
    order = np.lexsort(columns)  # (stable)
    differs = np.ones(m, dtype=bool)
    differs[1:] = np.any([c[order][1:] != c[order][:-1] for c in columns], axis=0)
    rank = np.maximum.accumulate(np.where(differs, np.arange(m), 0))
    alone = differs & np.append(differs[1:], True)
    want = np.concatenate([np.flatnonzero(~alone), np.flatnonzero(alone)])
    assert int(res.active) == int((~alone).sum()) > 0
    assert np.array_equal(got_rank, rank[want]) and np.array_equal(got_suf, lanes[order][want])
