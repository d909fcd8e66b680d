"""Seeded input texts shared by the oracle tests and the GPU parity tests (numpy PCG64, portable)."""
import numpy as np

SEP = 0xFFFF


def random_text(n, sigma, seed, sep_every=50):
    """n uint16 symbols over an alphabet of `sigma` values spread over [0, 65535] (0 and the maximum included),
    with separators 0xFFFF about every `sep_every` symbols: the shape of the reference's random fixtures
    (src/test_query.cu:317-331)."""
    rng = np.random.default_rng(seed)
    if sigma == 65536:
        alpha = np.arange(65536, dtype=np.uint64)
    else:
        alpha = (np.arange(sigma, dtype=np.uint64) * 65535) // max(sigma - 1, 1)
    T = alpha[rng.integers(0, len(alpha), size=n)].astype(np.uint16)
    if sep_every:
        T[rng.random(n) < 1.0 / sep_every] = SEP
    return T


def periodic(k=3000, a=3, b=7):
    return np.array([b if i % 2 else a for i in range(k)], dtype=np.uint16)


def fibonacci_word(min_len=2500):
    fib, prev = [1], [0]
    while len(fib) < min_len:
        fib, prev = fib + prev, fib
    return np.array(fib, dtype=np.uint16)


def hand_cases():
    """Texts of the reference's edge cases (src/test_query.cu:374-392) plus tail-rule corner cases."""
    cases = [
        [0, 0, 0, 0], [5, 3, 5, 0], [9, 8, 7], [3, 4, 5], [65535, 1, 65535, 1, 65535], [65535, 65535],
        [0], [7], [0, 0], [1, 0], [0, 1], [0, 0, 0], [0, 0, 0, 0, 0], [0] * 9, [0] * 17, [5, 0, 0, 0, 0, 5, 0, 0, 0],
        [5, 0, 0, 0, 5, 0, 0, 0], [1, 2, 3, 4, 1, 2, 3, 4, 1, 2, 3, 4], [1, 2, 3, 0, 0, 0, 0, 1, 2, 3, 0, 0, 0],
        [2, 1, 0, 0, 0, 0, 0, 0, 0, 0, 2, 1, 0, 0, 0, 0], list(range(20)), list(range(20, 0, -1)),
        [4] * 33, [0, 0, 0, 0, 0, 0, 0, 0, 1], [1, 0, 0, 0, 0, 0, 0, 0, 0],
    ]
    return [np.array(c, dtype=np.uint16) for c in cases]


def zero_tail_corner(n=5000, ell=4, seed=9):
    """Random text over a tiny alphabet ending in a run of zeros: the missing-terminator corner case
    (dataset/make-corner-case.py) whose expected first entries are n-1, n-2, ..., n-ell."""
    rng = np.random.default_rng(seed)
    T = rng.integers(0, 3, size=n).astype(np.uint16)
    T[-(ell + 3):] = 0
    return T


def fixture_suite():
    """(name, text) pairs used for golden vectors and parity."""
    out = []
    i = 0
    for n in (1, 2, 3, 15, 16, 17, 1000, 8000):
        for sigma in (2, 3, 4, 16, 256, 65536):
            out.append((f"rand_n{n}_s{sigma}", random_text(n, sigma, 1000 + i)))
            i += 1
    out.append(("periodic_ab", periodic()))
    out.append(("fibonacci", fibonacci_word()))
    out.append(("zero_tail", zero_tail_corner()))
    for k, c in enumerate(hand_cases()):
        out.append((f"hand_{k}", c))
    return out


def text_with_shared_codes(n, repeats, seed):
    """n random token ids into which strings of rare symbols are planted: for every r in `repeats`, r times the same three
    symbols of their own followed by one of two neighbouring symbols, the larger one first more often than not. Sorted by arithmetic
    codes of 32 bits, all r of them share one code as long as (r / n)^3 is far below 2^-32 times the symbols of the alphabet:
    runs of that length, out of order as they stand; each next to one planted the same way with a single string."""
    rng = np.random.default_rng(seed)
    T = rng.integers(1, 40000, n).astype(np.uint16)
    slots = rng.permutation(n // 5 - 2)
    at = 0
    for i, r in enumerate(repeats):
        for mixed in (0, 1):
            base = 50000 + 16 * (2 * i + mixed)
            for k in range(r):
                p = 5 * int(slots[at])
                at += 1
                T[p:p + 4] = [base, base + 1, base + 2, base + 4 - (mixed and int(rng.integers(0, 2)))]
    T[-2:] = 0
    return T


def text_of_phrases(n, phrases, lo, hi, seed):
    """n token ids made of `phrases` different sequences of lo to hi random ids each, drawn with Zipf(0.8) shares: symbols are rare and
    their successors few, so that the shares of single symbols say little about the strings that occur."""
    rng = np.random.default_rng(seed)
    ln = rng.integers(lo, hi + 1, phrases)
    start = np.cumsum(ln) - ln
    ids = rng.integers(1, 50000, int(ln.sum())).astype(np.uint16)
    share = np.arange(1, phrases + 1) ** -0.8
    draws = rng.choice(phrases, n // lo + 1, p=share / share.sum())
    at = np.repeat(start[draws] - (np.cumsum(ln[draws]) - ln[draws]), ln[draws]) + np.arange(int(ln[draws].sum()))
    return ids[at[:n]]


def text_of_shared_records(n, records, seed):
    """Records of four symbols: three that belong to the record's kind (`records` kinds) and one of 5000 values. All suffixes
    that start a record of one kind share an arithmetic code of 32 bits once (4 * records)^3 is near 2^32 / 4."""
    rng = np.random.default_rng(seed)
    kind = rng.integers(0, records, n // 4 + 1)
    T = np.stack([kind + 300, kind + 3000, kind + 6000, rng.integers(30000, 35000, kind.size)], axis=1)
    return T.reshape(-1)[:n].astype(np.uint16)


def text_with_repeated_strings(n, repeats, followers, end, seed):
    """n random token ids with four symbols planted r times for every r in `repeats`, each time followed by one of `followers` strings of
    four symbols (two of which differ in their last one only): runs of one string that are told apart by the next four symbols, into
    runs that are long again where r / followers is. `end`: the text ends in the planted string and as many zeros, which tie
    with the padding of a string that runs off the text."""
    rng = np.random.default_rng(seed)
    T = rng.integers(300, 60000, n).astype(np.uint16)
    slots = rng.permutation(n // 9 - 2)
    at = 0
    for i, r in enumerate(repeats):
        for k in range(r):
            p = 9 * int(slots[at])
            at += 1
            f = int(rng.integers(0, followers))
            T[p:p + 8] = [i, i, i + 1, i, 7, 5, f // 2, f % 2]
    if end:
        T[-4 - end:] = 0
        T[-4 - end:-end] = [0, 0, 1, 0]
    return T


def text_of_copies(n, symbols, seed):
    """n symbols below `symbols` into which passages are copied, several times over and over each other, some with a few symbols changed;
    every third text ends in zeros, every third in a copy of its start."""
    rng = np.random.default_rng(seed)
    T = rng.integers(0, symbols, n).astype(np.uint16)
    for _ in range(int(rng.integers(2, 12))):
        length = int(rng.integers(4, n // 3))
        src = int(rng.integers(0, n - length))
        passage = T[src:src + length].copy()
        for _ in range(int(rng.integers(1, 5))):
            dst = int(rng.integers(0, n - length))
            T[dst:dst + length] = passage
            if rng.random() < 0.5:
                at = dst + rng.integers(0, length, 3)
                T[at] = rng.integers(0, symbols, 3)
    if seed % 3 == 0:
        T[-int(rng.integers(1, 20)):] = 0
    elif seed % 3 == 1:
        T[n - n // 5:] = T[:n // 5]
    return T


SHORT_TEXTS = [(1, 1, 1), (5, 2, 1), (16, 60000, 4), (17, 2, 3), (513, 1, 2), (700, 60000, 1), (1025, 1, 1), (1025, 2, 4), (1500, 60000, 3)]


def short_text(n, sigma):
    """A text for the sort of short texts: a repeat and a run, so that more suffixes are tied than one workgroup takes to the end where
    n > 1000 (and all of them where sigma = 1), zeros at the end."""
    rng = np.random.default_rng(n + sigma)
    T = rng.integers(0, sigma, n).astype(np.uint16)
    T[n // 2:n // 2 + n // 4] = T[:n // 4]
    T[n // 8:n // 8 + n // 3] = T[0]
    T[n - n // 40:] = 0
    return T


def chains_text(kind, n):
    """Independent symbols around runs and stretches of one period, whose suffixes are all that is tied after a generation or two."""
    rng = np.random.default_rng(n)
    T = rng.integers(20, 60000, n).astype(np.uint16)
    if kind in ("rising", "falling", "two runs", "mixed"):
        T[n // 8:n // 8 + n // 6] = 17
        T[n // 8 + n // 6] = 1 if kind == "falling" else 50000
    if kind == "two runs":  # of one token: a group of two stretches, which the doubling goes on with
        T[n // 2:n // 2 + n // 7] = 17
    if kind in ("period", "mixed"):
        T[n // 2:n // 2 + n // 4] = np.resize(rng.integers(20, 60000, 7), n // 4)
    if kind == "mixed":
        T[9 * n // 10:9 * n // 10 + n // 20] = np.resize(rng.integers(20, 60000, 3), n // 20)
    if kind == "long period":  # looked at once ctx has reached it
        T[n // 4:n // 4 + n // 3] = np.resize(rng.integers(20, 60000, 30), n // 3)
    if kind == "end":  # the text ends inside the run
        T[-(n // 5):] = 30
    if kind == "period at the end":
        T[-(n // 5):] = np.resize(rng.integers(20, 60000, 7), n // 5)
    return T


CHAINS = ["rising", "falling", "two runs", "period", "mixed", "long period", "end", "period at the end"]


def text_of_undecided_copies(length):
    """A passage of `length` symbols three times, at residues 0, 4 and 0 modulo 8, the first eight symbols from each of its places 4, 12, 20, ...
    on once more in front of it, and an unrelated passage twice (so that groups have fewer than three members on average).
    In a sort that settles copies from anchors eight symbols apart, some pairs of the passage's copies are told apart by one record;
    for others every anchor says eight symbols and no more, and a comparison goes through the whole passage step by step."""
    rng = np.random.default_rng(length)
    M = rng.integers(100, 60000, length).astype(np.uint16)
    twice = rng.integers(100, 60000, 4000).astype(np.uint16)
    parts = []
    for o in range(4, length - 8, 8):
        parts += [M[o:o + 8], rng.integers(100, 60000, 3).astype(np.uint16)]
    at = sum(p.size for p in parts)
    for residue, end in ((0, 50), (4, 40), (0, 30)):
        gap = rng.integers(100, 60000, (residue - at) % 8).astype(np.uint16)
        parts += [gap, M, np.array([end], dtype=np.uint16)]
        at += gap.size + length + 1
    for _ in range(2):
        parts += [rng.integers(100, 60000, 20).astype(np.uint16), twice]
    return np.concatenate(parts + [rng.integers(100, 60000, 20).astype(np.uint16)])


def text_of_an_undecided_group(copies):
    """A passage of 24 symbols once on its own and `copies` times in front of another one of 160, the blocks of which (the first eight symbols from
    each of its places 4, 12, 20, ... on) stand in the text once more; and an unrelated passage twice. The members of a group of the short
    passage that go on with the long one differ from the first in the same way, and it takes two of them a step for every eight symbols of the
    long one to be told apart."""
    rng = np.random.default_rng(copies)
    short, long, twice = (rng.integers(100, 60000, k).astype(np.uint16) for k in (24, 160, 250 * copies))
    parts = [short, rng.integers(100, 60000, 8).astype(np.uint16)]
    for o in range(4, long.size - 8, 8):
        parts += [long[o:o + 8], rng.integers(100, 60000, 3).astype(np.uint16)]
    at = sum(p.size for p in parts)
    for c in range(copies):
        gap = rng.integers(100, 60000, 8 + (4 * c - at) % 8).astype(np.uint16)
        parts += [gap, short, long]
        at += gap.size + short.size + long.size
    for _ in range(2):
        parts += [rng.integers(100, 60000, 20).astype(np.uint16), twice]
    return np.concatenate(parts + [rng.integers(100, 60000, 20).astype(np.uint16)])


def written_text(n, words, seed, letters=26):
    """n byte symbols of words of 1 to 9 lower-case letters, the first ones the most frequent, a space between words."""
    rng = np.random.default_rng(seed)
    vocabulary = [rng.integers(97, 97 + letters, int(rng.integers(1, 10))).tolist() + [32] for _ in range(words)]
    ids = np.minimum(rng.zipf(1.3, n), words) - 1  # (a word is two symbols at least)
    text = [symbol for i in ids[:n // 2 + 1] for symbol in vocabulary[i]]
    return np.array(text[:n], dtype=np.uint16)


def text_of_planted_strings(n, symbols, repeats, seed):
    """n independent symbols, 1 to `symbols` (or 0 to 3, of two bits), among them strings that come repeats[i] times each, at multiples of 16, their first symbols spread over the whole alphabet: of
    four symbols, or of 16 where the alphabet has four letters."""
    rng = np.random.default_rng(seed)
    T = rng.integers(1, symbols + 1, n).astype(np.uint16)
    places = 16 * rng.permutation(n // 16 - 1)[:sum(repeats)]
    for i, times in enumerate(repeats):
        at, places = places[:times], places[times:]
        if symbols > 4:
            string = np.concatenate([[1 + (2 * i + 1) * (symbols - 1) // (2 * len(repeats))], rng.integers(1, symbols + 1, 3)])
        else:
            string = np.concatenate([[1 + i * 16 // len(repeats) // 4, 1 + i * 16 // len(repeats) % 4], rng.integers(1, symbols + 1, 14)])
        T[at[:, None] + np.arange(string.size)] = string
    return T if symbols > 4 else T - np.uint16(1)


def marked_text(n, values, kind, seed):
    """n symbols over `values` values, zero among them: independent ones with copies, or words with marks in between, and what `kind` says (a period over a
    fiftieth of it, zeros here and there and at the end, a phrase that comes 700 times and ends the text inside)."""
    rng = np.random.default_rng(seed)
    if kind == "copies":
        T = rng.integers(0, values, n).astype(np.uint16)
        for k in range(10):
            T[k * n // 10 + n // 20:k * n // 10 + n // 20 + n // 50] = T[k * n // 10:k * n // 10 + n // 50]
    else:
        T = np.maximum(written_text(n, 1500, seed, min(values - 1, 26)).astype(np.int64) - 96, 0)  # (the space is zero)
        marks = rng.permutation(n // 20)[:n // 40] * 20
        T[marks] = rng.integers(0, values, marks.size)
    if kind == "period":
        T[n // 3:n // 3 + n // 50] = np.resize(T[:11], n // 50)
    elif kind == "zeros":
        for at in rng.permutation(n // 40 - 1)[:n // 400]:
            T[40 * at:40 * at + int(rng.integers(3, 36))] = 0
        T[-30:] = 0
    elif kind == "end":
        phrase = rng.integers(1, values, 24)
        for at in rng.permutation(n // 64 - 1)[:700]:
            T[64 * at:64 * at + 24] = phrase
        T[-16:] = phrase[:16]
    T[:values] = np.arange(values)
    return T.astype(np.uint16)
