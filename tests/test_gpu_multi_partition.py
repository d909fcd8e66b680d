"""The exported stage kernels composed into the reference's multi-partition pipeline on the GPU (tests/multi_partition.py):
partitions exchange ranks only through messages; the suffix array must equal the oracle's."""
import ctypes as C

import numpy as np
import pytest

import multi_partition
import oracle_lib
import texts
from test_gpu_messages import DevArray

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import torch
    from cascade_amd import _native
    assert torch.cuda.is_available()
    to_t = {np.dtype(np.uint64): np.int64, np.dtype(np.uint32): np.int32, np.dtype(np.uint16): np.int16, np.dtype(np.uint8): np.uint8}
    back = {np.dtype(np.int64): np.uint64, np.dtype(np.int32): np.uint32, np.dtype(np.int16): np.uint16, np.dtype(np.uint8): np.uint8}

    def to_dev(a):
        a = np.ascontiguousarray(a)
        return DevArray(torch.from_numpy(a.view(to_t[a.dtype])).cuda())

    def to_host(d):
        torch.cuda.synchronize()
        a = d.t.cpu().numpy()
        return a.view(back[a.dtype])

    return _native.load(), to_dev, to_host


def steps_handle(lib, key_words):
    """For multi_partition.build_sa: a handle made for the steps (csa_create_steps) with exactly the largest partition's
    capacity, the tightest the floor plan admits: a step that needs a byte more than csa_step_bytes_per_suffix fails."""
    def make(max_part_sz):
        h = C.c_void_p()
        assert lib.csa_create_steps(max_part_sz, key_words, C.byref(h)) == 0, lib.csa_last_error()
        return h
    return make


@pytest.mark.parametrize("p,key_words,sorted_join,steps", [(3, 1, False, False), (16, 1, True, False), (33, 2, False, False),
                                                           (3, 1, False, True), (16, 2, False, True), (40, 1, False, True),
                                                           (9, 3, False, True), (16, 4, False, True), (5, 4, False, False)])
def test_partitions_that_only_exchange_messages_build_the_oracles_suffix_array(gpu, p, key_words, sorted_join, steps):
    """steps = False: numpy glue between the exported stage kernels; True: each partition step is one call of
    csa_sort_init_dev / csa_sort_rerank_dev."""
    lib, to_dev, to_host = gpu
    n = 120000
    T = texts.random_text(n, 4, 7 * p, sep_every=0)
    T[30000:70000] = T[:40000]  # a long repeat: many generations, forwarded pills
    T[-9:] = 0
    log = []
    h = C.c_void_p()
    assert lib.csa_create(n, 1, C.byref(h)) == 0
    try:
        print(f"  multi-partition n={n} p={p} key_words={key_words} steps={steps}", flush=True)
        sa, gens = multi_partition.build_sa(lib, to_dev, to_host, T, p, key_words=key_words, log=log,
                                            join_handle=h if sorted_join else None,
                                            step_handle=steps_handle(lib, key_words) if steps else None)
    finally:
        lib.csa_destroy(h)
    want, _ = oracle_lib.prefix_doubling(T, key_words)
    assert np.array_equal(sa, want)
    assert gens >= 10 and sum(step[5] for step in log if step[0] >= 1) > 0


def pinned_host_buf(nbytes):
    """uint8 numpy view of freshly pinned host memory (the view keeps the tensor alive)."""
    import torch
    return torch.empty(max(int(nbytes), 1), dtype=torch.uint8, pin_memory=True).numpy()


@pytest.mark.parametrize("p,key_words,chunk_cap", [(3, 1, 4096), (16, 2, 8192), (40, 1, 4096), (9, 4, 4096), (1, 1, 32768)])
def test_slab_shaped_entries_from_pinned_host_slabs_build_the_oracles_suffix_array(gpu, p, key_words, chunk_cap):
    """The three members as the reference's dispatcher calls them (src/GPU_SACA.cu:1579-1580, 2356): every partition step takes
    the partition as pinned host slabs of ragged sizes (upload, device step, download inside csa_sort_init_slabs /
    csa_sort_rerank_slabs), and csa_scatter_slabs returns each partition's stretch of the output cut into disk blocks and
    edges. The file assembled from those pieces is the oracle's suffix array."""
    lib, to_dev, to_host = gpu
    n = 120000
    T = texts.random_text(n, 4, 11 * p, sep_every=0)
    T[30000:70000] = T[:40000]
    T[-9:] = 0
    log = []
    print(f"  slab entries n={n} p={p} key_words={key_words} chunk_cap={chunk_cap}", flush=True)
    sa, gens = multi_partition.build_sa(lib, to_dev, to_host, T, p, key_words=key_words, log=log, slab_handle=steps_handle(lib, key_words),
                                        host_buf=pinned_host_buf, chunk_cap=chunk_cap)
    per_suffix = int(lib.csa_step_bytes_per_suffix(key_words))
    assert per_suffix == {1: 48, 2: 65, 3: 76, 4: 84}[key_words]
    assert multi_partition.build_sa.high_water <= per_suffix * (n + 255)  # (the partition's size is rounded up to 256 suffixes)
    want, _ = oracle_lib.prefix_doubling(T, key_words)
    assert np.array_equal(sa, want)
    assert gens >= 10 and (p == 1 or sum(step[5] for step in log if step[0] >= 1) > 0)


def test_slab_shaped_entries_report_what_the_device_entries_report(gpu):
    """The same pipeline through csa_sort_*_dev and through csa_sort_*_slabs: cohort, survivors, messages and pills agree in
    every generation of every partition."""
    lib, to_dev, to_host = gpu
    from cascade_amd import workloads
    T = workloads.generate(3, 200000)
    n, p = T.size, 12
    logs = []
    for mode in ("dev", "slabs"):
        log = []
        print(f"  {mode} entries n={n} p={p}", flush=True)
        make = steps_handle(lib, 1)
        kw = {"step_handle": make} if mode == "dev" else {"slab_handle": make, "host_buf": pinned_host_buf, "chunk_cap": 8192}
        sa, _ = multi_partition.build_sa(lib, to_dev, to_host, T, p, log=log, seed=5, **kw)
        assert np.array_equal(sa, oracle_lib.prefix_doubling(T, 1)[0])
        logs.append(log)
    assert logs[0] == logs[1]


def test_slab_entries_refuse_slabs_that_do_not_make_up_the_partition(gpu):
    lib, _, _ = gpu
    from cascade_amd import _native
    h = C.c_void_p()
    assert lib.csa_create(10000, 1, C.byref(h)) == 0
    try:
        pool = multi_partition.SlabPool(pinned_host_buf, 4096, 1)
        arr, slab_c, _ = pool.assemble([(0, 4096), (4096, 1000)])
        end, act = np.zeros(3, dtype=np.uint32), C.c_uint64(0)
        # sizes that do not add up to the partition, a slab beyond chunk_cap, a partition beyond the handle
        assert lib.csa_sort_init_slabs(h, arr, slab_c, 6000, 1, 3, 4096, end.ctypes.data, C.byref(act), None) == _native.CSA_ERR_ARG
        assert b"slabs hold" in lib.csa_last_error()
        assert lib.csa_sort_init_slabs(h, arr, slab_c, 5096, 1, 3, 4000, end.ctypes.data, C.byref(act), None) == _native.CSA_ERR_ARG
        assert lib.csa_sort_init_slabs(h, arr, slab_c, 20000, 1, 3, 4096, end.ctypes.data, C.byref(act), None) == _native.CSA_ERR_ARG
        # slabs that overlap although their sizes add up
        arr3, c3, _ = pool.assemble([(0, 3000), (2000, 2096)])
        assert lib.csa_sort_init_slabs(h, arr3, c3, 5096, 1, 3, 4096, end.ctypes.data, C.byref(act), None) == _native.CSA_ERR_ARG
        assert b"starts at suffix" in lib.csa_last_error()
        # an inbox that the slabs do not carry in full
        assert lib.csa_sort_rerank_slabs(h, arr, slab_c, 5096, 77, 8, 3, 4096, end.ctypes.data, C.byref(act), None) == _native.CSA_ERR_ARG
        assert b"inbox" in lib.csa_last_error()
        # a scatter whose chunks cannot carry the output: chunk_cap not a multiple of 4096 suffixes
        arr2, c2, bufs = pool.assemble([(0, 3000), (3000, 2096)])
        for b in bufs:
            b["key"].view(np.uint32)[:4096] = 0
        assert lib.csa_scatter_slabs(h, arr2, c2, 5096, 0, 3000, None) == _native.CSA_ERR_ARG
    finally:
        lib.csa_destroy(h)


def _shape(name):
    from cascade_amd import workloads
    if name == "one_symbol":       # one group until the very end; every pivot equal, so all but one partition are empty
        return np.full(50000, 7, dtype=np.uint16)
    if name == "period_7":         # groups of n / 7 members for log2(n) generations
        return np.tile(np.array([3, 1, 4, 1, 5, 9, 2], dtype=np.uint16), 9000)
    if name == "zipf_duplicates":  # the headline construction, scaled down: long duplicated documents
        return workloads.generate(3, 400000)
    if name == "adversarial":      # a token run, a periodic stretch and Zipf text in one partition set
        return workloads.generate(5, 300000)
    raise KeyError(name)


@pytest.mark.parametrize("shape,p", [("one_symbol", 5), ("period_7", 9), ("zipf_duplicates", 300), ("adversarial", 64)])
def test_step_entries_on_hard_shapes(gpu, shape, p):
    """csa_sort_init_dev / csa_sort_rerank_dev per partition and generation, on texts whose groups stay large for many
    generations, with empty partitions and with hundreds of partitions."""
    lib, to_dev, to_host = gpu
    T = _shape(shape)
    n = T.size
    print(f"  step entries on {shape}: n={n} p={p}", flush=True)
    sa, gens = multi_partition.build_sa(lib, to_dev, to_host, T, p, step_handle=steps_handle(lib, 1))
    want, _ = oracle_lib.prefix_doubling(T, 1)
    assert np.array_equal(sa, want), (shape, gens)
    if shape == "one_symbol":
        assert np.array_equal(sa, np.arange(n - 1, -1, -1, dtype=np.uint64))


@pytest.mark.parametrize("p,key_words,pivot_words,slabs", [(16, 1, 1, False), (7, 2, 2, True), (40, 4, 2, False)])
def test_the_references_own_predictor_gives_the_cohorts_and_pill_receipts_of_the_steps(gpu, tmp_path, p, key_words, pivot_words, slabs):
    """The reference's src/sa_structure.cpp (compiled from its one source file into oracle/_ref) predicts a run from the
    finished suffix array, the key and pivot widths and the partition sizes: every generation's active-set size, every
    query's look-back, the messages before any is withheld from a retired recipient. 150 000 symbols with long repeats in
    7 to 40 partitions through the device and the slab entries: the steps must have had exactly those cohorts and exactly
    that many members joined by a pill (csa_step_result.pills), summed over the partitions, and emit that many messages in
    generation 0 and never more later."""
    import os
    if not os.path.exists(oracle_lib.SA_STRUCTURE):
        pytest.skip("oracle/_ref/sa_structure is not built (make -C oracle where the reference tree is present)")
    lib, to_dev, to_host = gpu
    rng = np.random.default_rng(p)
    T = rng.integers(0, 5, 150000).astype(np.uint16)
    T[90000:130000] = T[10000:50000]
    T[140000:141000] = T[0]
    T[-11:] = 0
    log = []
    kw = {"slab_handle": steps_handle(lib, key_words), "host_buf": pinned_host_buf, "chunk_cap": 8192} if slabs else {
        "step_handle": steps_handle(lib, key_words)}
    print(f"  pipeline against sa_structure p={p} key_words={key_words} pivot_words={pivot_words} slabs={slabs}", flush=True)
    sa, _ = multi_partition.build_sa(lib, to_dev, to_host, T, p, key_words=key_words, pivot_words=pivot_words, seed=p, log=log, **kw)
    want, _ = oracle_lib.prefix_doubling(T, 1)
    assert np.array_equal(sa, want)
    ours, theirs = multi_partition.structure_of_a_pipeline_run(T, p, key_words, pivot_words, p, log, multi_partition.build_sa.pill_receipts,
                                                               tmp_path)
    assert ours["cohorts"] == theirs["cohorts"], (ours, theirs)
    assert ours["pill_receipts"] == theirs["pill_receipts"], (ours, theirs)
    assert ours["messages"][0] == theirs["messages"][0] and all(a <= b for a, b in zip(ours["messages"], theirs["messages"]))
    assert len(ours["cohorts"]) >= 10 and sum(ours["pill_receipts"]) > 0


@pytest.mark.parametrize("key_words,long_runs", [(1, True), (2, False), (2, True), (3, True), (4, False), (4, True), (2, "few"), (4, "few"), (2, "many"), (4, "many")])
def test_runs_of_one_first_word_in_order(gpu, key_words, long_runs):
    """csa_sort_init_dev with runs of one first word at the edges of what is sorted in place, against a sort of whole keys."""
    import message_cases
    lib, to_dev, to_host = gpu
    print(f"  runs of one first word: key_words={key_words} long_runs={long_runs}", flush=True)
    message_cases.check_runs_of_first_words(lib, to_dev, to_host, steps_handle(lib, key_words), key_words, long_runs)


def test_random_pipelines_through_the_step_entries(gpu):
    """Random texts (tiny alphabets, long repeats, zero tails), 1 to 200 partitions, all four key widths: every step
    passes the reference's validators inside the harness and the suffix array is the oracle's."""
    lib, to_dev, to_host = gpu
    rng = np.random.default_rng(99)
    for case in range(40):
        n = int(rng.integers(50, 30000))
        sigma = int(rng.choice([1, 2, 3, 5, 40, 65536]))
        T = rng.integers(0, sigma, n).astype(np.uint16)
        if case % 3 == 1 and n > 200:
            length = int(rng.integers(10, n // 2))
            T[n - length:] = T[:length]
        if case % 3 == 2:
            T[-int(rng.integers(1, 30)):] = 0
        p = int(rng.choice([1, 2, 3, 7, 16, 50, 200]))
        key_words = 1 + case % 4
        print(f"  random pipeline case={case} n={n} sigma={sigma} p={p} key_words={key_words}", flush=True)
        # half of the cases through the slab-shaped entries; the handle is sized exactly for the largest partition
        kw = {"step_handle": steps_handle(lib, key_words)} if (case // 4) % 2 == 0 else {
            "slab_handle": steps_handle(lib, key_words), "host_buf": pinned_host_buf, "chunk_cap": 4096}
        sa, _ = multi_partition.build_sa(lib, to_dev, to_host, T, p, key_words=key_words, seed=case, **kw)
        want, _ = oracle_lib.prefix_doubling(T, 1)
        assert np.array_equal(sa, want), (case, n, sigma, p, key_words)
