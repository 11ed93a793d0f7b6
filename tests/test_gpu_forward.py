"""GPU parity tests of bm_moe_forward, the one entry for any number of tokens: each of its three paths (per slot, grouped
by expert, the grouped GEMM) gives the oracle's layer output bit for bit on the same seeded inputs, so the choice among
them by batch size changes no bit; a forced path takes its own launches and the automatic choice follows the crossovers; ids that name no
expert add nothing."""
import ctypes as C

import numpy as np
import pytest

import bloomery_amd as bm
import ora
from common import normal_f32
from test_gpu_decode import Layer, assert_f32, gpu, route  # noqa: F401  (gpu: module fixture)

pytestmark = pytest.mark.gpu

PATHS = ((bm.PATH_PER_SLOT, "per slot"), (bm.PATH_GROUPED, "grouped"), (bm.PATH_GEMM, "gemm"))


class _KernelNode(C.Structure):  # hipKernelNodeParams
    _fields_ = [("threads", C.c_uint32 * 3), ("extra", C.c_void_p), ("func", C.c_void_p), ("blocks", C.c_uint32 * 3), ("params", C.c_void_p),
                ("lds", C.c_uint32)]


def launches(gpu, enqueue):
    """The workgroups' thread counts of the launches that `enqueue` makes, in order: captured on the context's stream, not run."""
    with open("/proc/self/maps") as f:
        hip = C.CDLL(next(line.split()[-1] for line in f if "libamdhip64.so" in line))  # the runtime that the library has loaded
    graph, count = C.c_void_p(), C.c_size_t(0)
    assert hip.hipStreamBeginCapture(C.c_void_p(gpu.stream()), 1) == 0  # (thread-local)
    try:
        enqueue()
    finally:
        assert hip.hipStreamEndCapture(C.c_void_p(gpu.stream()), C.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, C.byref(count)) == 0
    nodes, threads = (C.c_void_p * count.value)(), []
    assert hip.hipGraphGetNodes(graph, nodes, C.byref(count)) == 0
    for n in nodes:
        p = _KernelNode()
        assert hip.hipGraphKernelNodeGetParams(C.c_void_p(n), C.byref(p)) == 0
        threads.append(p.threads[0])
    assert hip.hipGraphDestroy(graph) == 0
    return threads


def route_taken(gpu, enqueue):
    """Which launches a step of two Q8_K stacks makes: the per-slot step's two, the grouped step's, which begin with the tables (a workgroup of
    1024 threads), or slot by slot through launches of their own, which begin with the quantizer."""
    t = launches(gpu, enqueue)
    return "per slot" if len(t) == 2 else "tiles" if t[0] == 1024 else "slot by slot" if len(t) == 5 else t


@pytest.mark.parametrize("types,hidden,ff,n_experts,top_k,m", (
    ((bm.Q4_K, bm.Q4_K, bm.Q6_K), 2048, 768, 12, 8, 19),     # the headline layer's rows
    ((bm.Q5_K, bm.Q5_K, bm.Q4_K), 512, 512, 5, 3, 40),
    ((bm.IQ2_XXS, bm.IQ2_XXS, bm.IQ2_XXS), 1024, 512, 6, 4, 9),  # Q8_K columns on both sides
    ((bm.Q4_K, bm.Q4_K, bm.IQ2_XXS), 512, 768, 4, 2, 33),    # the two column forms in one layer
    ((bm.IQ4_XS, bm.IQ4_XS, bm.Q3_K), 512, 512, 5, 3, 25),   # the added types through the GEMM path as well
    ((bm.IQ3_XXS, bm.IQ3_XXS, bm.Q6_K), 768, 256, 4, 2, 18),
    ((bm.IQ2_XXS, bm.IQ2_XXS, bm.IQ2_XXS), 512, 512, 40, 4, 6),  # no more slots than experts, Q8_K columns on both sides: the
    ((bm.IQ4_XS, bm.IQ4_XS, bm.Q3_K), 512, 256, 64, 3, 7),       # grouped path's launches go slot by slot
))
def test_every_path_gives_the_oracles_bits(gpu, types, hidden, ff, n_experts, top_k, m):
    L = Layer(gpu, types, hidden, ff, n_experts, 5100 + hidden)
    rng = np.random.default_rng(5101)
    x, resid = normal_f32(rng, (m, hidden)), normal_f32(rng, (m, hidden))
    ids, wts = route(rng, m, n_experts, top_k)
    want_y, _ = L.oracle(x, ids, wts, top_k)
    want = (want_y.reshape(m, hidden) + resid).astype(np.float32).reshape(-1)
    xd, sel, wd, rd = gpu.upload(x, np.float32), gpu.upload(ids, np.uint32), gpu.upload(wts, np.float32), gpu.upload(resid, np.float32)
    y = gpu.buffer(np.float32, m * hidden)
    sc = gpu.scratch(types[0], types[2], hidden, ff, n_experts, top_k, 64)
    gpu.fault_clear()
    try:
        for path, name in PATHS:
            sc.set_path(path)
            assert sc.path_for(m) == path
            for rep in range(2):  # the scratch is reused as it stands
                y.fill_bytes(0xFF)
                gpu.enqueue_moe_forward(sc, L.dg, L.du, L.dd, xd, sel, wd, rd, m, y)
                assert_f32(y.download(), want, f"{name}, call {rep}")
            # fewer tokens after more, over the same scratch
            y.fill_bytes(0xFF)
            gpu.enqueue_moe_forward(sc, L.dg, L.du, L.dd, xd, sel, wd, rd, 3, y)
            assert_f32(y.download()[:3 * hidden], want[:3 * hidden], f"{name}, three tokens")
        assert gpu.fault() == (bm.FAULT_NONE, 0)
    finally:
        sc.free()
        for b in (xd, sel, wd, rd, y):
            b.free()
        L.free()


@pytest.mark.parametrize("m", (19, 20))
def test_per_slot_step_on_either_side_of_its_own_launches(gpu, m):
    """Stacks on Q8_K columns whose rows are 6.7 MB an expert: 20 slots ask for 128 MB, from where the per-slot step quantizes its columns in
    launches of their own with three slots a token and more (with one, as here, from 200 MB: test_a_forced_path_takes_its_own_launches). One
    slot is served elsewhere and one names no expert; neither adds anything."""
    hidden, ff, n_experts, top_k = 2048, 2048, 8, 1
    L = Layer(gpu, (bm.IQ4_XS, bm.IQ4_XS, bm.IQ4_XS), hidden, ff, n_experts, 5200, cheap=True)
    rng = np.random.default_rng(5201)
    x, resid = normal_f32(rng, (m, hidden)), normal_f32(rng, (m, hidden))
    ids, wts = route(rng, m, n_experts, top_k)
    want_y, _ = L.oracle(x, ids, wts, top_k)
    want = (want_y.reshape(m, hidden) + resid).astype(np.float32)
    ids[2], ids[5] = bm.HOST_SLOT, n_experts
    want[[2, 5]] = resid[[2, 5]]
    xd, sel, wd, rd = gpu.upload(x, np.float32), gpu.upload(ids, np.uint32), gpu.upload(wts, np.float32), gpu.upload(resid, np.float32)
    y = gpu.buffer(np.float32, m * hidden).fill_bytes(0xFF)
    sc = gpu.scratch(bm.IQ4_XS, bm.IQ4_XS, hidden, ff, n_experts, top_k, 32)
    gpu.fault_clear()
    try:
        assert sc.path_for(m) == bm.PATH_PER_SLOT
        for _ in range(2):
            gpu.enqueue_moe_forward(sc, L.dg, L.du, L.dd, xd, sel, wd, rd, m, y)
            assert_f32(y.download(), want.reshape(-1), "y")
        assert gpu.fault()[1] == 1 << bm.SITE_EXPERT_ID
    finally:
        gpu.fault_clear()
        sc.free()
        for b in (xd, sel, wd, rd, y):
            b.free()
        L.free()


@pytest.mark.parametrize("types,hidden,ff,n_experts,top_k,m,auto,grouped", (
    ((bm.IQ4_XS, bm.IQ4_XS, bm.IQ4_XS), 2048, 3072, 8, 1, 19, "per slot", "tiles"),      # 191 MB asked for
    ((bm.IQ4_XS, bm.IQ4_XS, bm.IQ4_XS), 2048, 3072, 8, 1, 20, "slot by slot", "tiles"),  # 201 MB
    ((bm.Q3_K, bm.Q3_K, bm.IQ3_XXS), 2048, 2048, 8, 3, 8, "per slot", "tiles"),          # 125 MB, three slots a token
    ((bm.Q3_K, bm.Q3_K, bm.IQ3_XXS), 2048, 2048, 8, 3, 9, "slot by slot", "tiles"),      # 141 MB
    ((bm.IQ4_XS, bm.IQ4_XS, bm.IQ4_XS), 2048, 3840, 4, 2, 21, "slot by slot", "tiles"),  # 526 MB, more slots than experts
    ((bm.IQ2_XXS, bm.IQ2_XXS, bm.IQ2_XXS), 1024, 512, 6, 4, 9, "per slot", "tiles"),
    ((bm.IQ2_XXS, bm.IQ2_XXS, bm.Q3_K), 512, 256, 27, 3, 9, "per slot", "slot by slot"),  # a slot an expert
    ((bm.IQ2_XXS, bm.IQ2_XXS, bm.Q3_K), 512, 256, 26, 3, 9, "per slot", "tiles"),
    ((bm.IQ3_XXS, bm.IQ3_XXS, bm.IQ4_XS), 512, 512, 64, 3, 24, "slot by slot", "tiles"),  # past the per-slot step's tokens
    ((bm.IQ2_XXS, bm.IQ2_XXS, bm.IQ2_XXS), 512, 512, 16, 4, 76, "slot by slot", "tiles"),  # nineteen slots an expert: what its tiles save
    ((bm.IQ2_XXS, bm.IQ2_XXS, bm.IQ2_XXS), 512, 512, 16, 4, 77, "tiles", "tiles"),
    ((bm.IQ4_XS, bm.IQ4_XS, bm.IQ4_XS), 4096, 1024, 4, 1, 74, "slot by slot", "tiles"),    # 495 MB
    ((bm.IQ4_XS, bm.IQ4_XS, bm.IQ4_XS), 4096, 1024, 4, 1, 75, "tiles", "tiles"),           # 501 MB
))
def test_a_forced_path_takes_its_own_launches(gpu, types, hidden, ff, n_experts, top_k, m, auto, grouped):
    """Stacks on Q8_K columns on both sides: the per-slot and the grouped path forced, and what the automatic choice puts in their place, as
    launches and in their outputs, with slots that are served elsewhere and refused ones."""
    L = Layer(gpu, types, hidden, ff, n_experts, 5210 + m, cheap=True)
    rng = np.random.default_rng(5211)
    x, resid = normal_f32(rng, (m, hidden)), normal_f32(rng, (m, hidden))
    ids, wts = route(rng, m, n_experts, top_k)
    wts[2, 0] = wts[m - 1, top_k - 1] = 0.0  # (the two slots that no expert takes below)
    want = (L.oracle(x, ids, wts, top_k)[0].reshape(m, hidden) + resid).astype(np.float32).reshape(-1)
    ids[2, 0], ids[m - 1, top_k - 1] = bm.HOST_SLOT, n_experts
    xd, sel, wd, rd = gpu.upload(x, np.float32), gpu.upload(ids, np.uint32), gpu.upload(wts, np.float32), gpu.upload(resid, np.float32)
    y = gpu.buffer(np.float32, m * hidden)
    sc = gpu.scratch(types[0], types[2], hidden, ff, n_experts, top_k, m)
    step = lambda: gpu.enqueue_moe_forward(sc, L.dg, L.du, L.dd, xd, sel, wd, rd, m, y)  # noqa: E731
    try:
        for path, takes in ((bm.PATH_AUTO, auto), (bm.PATH_PER_SLOT, "per slot"), (bm.PATH_GROUPED, grouped)):
            sc.set_path(path, 0, 4096)  # (the automatic choice among the two of them alone)
            assert route_taken(gpu, step) == takes, path
            gpu.fault_clear()
            for _ in range(2):
                y.fill_bytes(0xFF)
                step()
                assert_f32(y.download(), want, f"path {path}")
            assert gpu.fault()[1] == 1 << bm.SITE_EXPERT_ID
    finally:
        gpu.fault_clear()
        sc.free()
        for b in (xd, sel, wd, rd, y):
            b.free()
        L.free()


@pytest.mark.parametrize("types,hidden,ff,n_experts,top_k,m,mode,slots", (
    ((bm.IQ4_XS, bm.IQ4_XS, bm.IQ4_XS), 1792, 256, 2, 1, 31, bm.GEMM_EXACT, True),   # fifteen slots an expert: half the GEMM's time
    ((bm.IQ4_XS, bm.IQ4_XS, bm.IQ4_XS), 1792, 256, 2, 1, 31, bm.GEMM_FAST, True),    # below 96 tokens the exact order in this mode too
    ((bm.IQ4_XS, bm.IQ4_XS, bm.Q3_K), 512, 256, 4, 2, 99, bm.GEMM_EXACT, True),
    ((bm.IQ4_XS, bm.IQ4_XS, bm.Q3_K), 512, 256, 4, 2, 100, bm.GEMM_EXACT, False),
    ((bm.IQ3_XXS, bm.IQ3_XXS, bm.IQ2_XXS), 256, 512, 1, 1, 266, bm.GEMM_EXACT, True),
    ((bm.IQ3_XXS, bm.IQ3_XXS, bm.IQ2_XXS), 256, 512, 1, 1, 267, bm.GEMM_EXACT, False),
))
def test_few_slots_of_few_experts_go_slot_by_slot_in_the_gemms_place(gpu, types, hidden, ff, n_experts, top_k, m, mode, slots):
    """Stacks on Q8_K columns where the path is the GEMM's: on both sides of the line from which its launches run, in its exact order; a
    caller's own line or a forced path takes them at once. Outputs are the oracle's either way."""
    L = Layer(gpu, types, hidden, ff, n_experts, 5230 + m, cheap=True)
    rng = np.random.default_rng(5231)
    x, resid = normal_f32(rng, (m, hidden)), normal_f32(rng, (m, hidden))
    ids, wts = route(rng, m, n_experts, top_k)
    wts[2, 0] = wts[m - 1, top_k - 1] = 0.0  # (the two slots that no expert takes below)
    want = (L.oracle(x, ids, wts, top_k)[0].reshape(m, hidden) + resid).astype(np.float32).reshape(-1)
    ids[2, 0], ids[m - 1, top_k - 1] = bm.HOST_SLOT, n_experts
    xd, sel, wd, rd = gpu.upload(x, np.float32), gpu.upload(ids, np.uint32), gpu.upload(wts, np.float32), gpu.upload(resid, np.float32)
    y = gpu.buffer(np.float32, m * hidden)
    sc = gpu.scratch(types[0], types[2], hidden, ff, n_experts, top_k, m)
    step = lambda: gpu.enqueue_moe_forward(sc, L.dg, L.du, L.dd, xd, sel, wd, rd, m, y)  # noqa: E731
    gpu.set_gemm_mode(mode)
    try:
        ways = ((bm.PATH_AUTO, 0, slots), (bm.PATH_GEMM, 0, False), (bm.PATH_AUTO, 1, False))
        for path, line, takes in ways if mode == bm.GEMM_EXACT else ways[:1]:
            sc.set_path(path, 0, line)
            assert sc.path_for(m) == bm.PATH_GEMM
            assert (route_taken(gpu, step) == "slot by slot") == takes, (path, line)
            gpu.fault_clear()
            for _ in range(2):
                y.fill_bytes(0xFF)
                step()
                assert_f32(y.download(), want, f"path {path}, line {line}")
            assert gpu.fault()[1] == 1 << bm.SITE_EXPERT_ID
    finally:
        gpu.set_gemm_mode(bm.GEMM_EXACT)
        gpu.fault_clear()
        sc.free()
        for b in (xd, sel, wd, rd, y):
            b.free()
        L.free()


@pytest.mark.parametrize("m,top_k", ((8, 3), (7, 3), (6, 3), (20, 1)))
def test_rows_of_tokens_that_no_expert_takes_may_hold_anything(gpu, m, top_k):
    """A per-slot step of the automatic choice, in launches of its own (24 and 21 slots, 160 and 140 MB asked for) and in two: a row whose slots are all
    served elsewhere, or refused, is not read as numbers. It may hold NaN and infinities and raises nothing but the refused id; the
    other tokens' rows, one of them with some slots served elsewhere, are the oracle's."""
    hidden, ff, n_experts = 2048, 2048, 8
    L = Layer(gpu, (bm.IQ4_XS, bm.IQ4_XS, bm.IQ4_XS), hidden, ff, n_experts, 5200, cheap=True)
    rng = np.random.default_rng(5202)
    x, resid = normal_f32(rng, (m, hidden)), normal_f32(rng, (m, hidden))
    ids, wts = route(rng, m, n_experts, top_k)
    ids, wts = ids.reshape(m, top_k), wts.reshape(m, top_k)
    if top_k > 1:
        wts[4, :-1] = 0.0  # (the slots that are served elsewhere below)
    want_y, _ = L.oracle(x, ids, wts, top_k)
    want = (want_y.reshape(m, hidden) + resid).astype(np.float32)
    ids[4, :-1] = bm.HOST_SLOT
    ids[2], ids[m - 1] = bm.HOST_SLOT, bm.HOST_SLOT
    x[2], x[m - 1, 5] = np.nan, np.inf
    want[[2, m - 1]] = resid[[2, m - 1]]
    xd, wd, rd = gpu.upload(x, np.float32), gpu.upload(wts, np.float32), gpu.upload(resid, np.float32)
    y = gpu.buffer(np.float32, m * hidden)
    sc = gpu.scratch(bm.IQ4_XS, bm.IQ4_XS, hidden, ff, n_experts, top_k, 32)
    try:
        assert sc.path_for(m) == bm.PATH_PER_SLOT
        for refused in (False, True):
            if refused:
                ids[2] = n_experts
            sel = gpu.upload(ids, np.uint32)
            gpu.fault_clear()
            y.fill_bytes(0xFF)
            gpu.enqueue_moe_forward(sc, L.dg, L.du, L.dd, xd, sel, wd, rd, m, y)
            assert_f32(y.download(), want.reshape(-1), f"refused {refused}")
            assert gpu.fault()[1] == (1 << bm.SITE_EXPERT_ID if refused else 0)
            sel.free()
    finally:
        gpu.fault_clear()
        sc.free()
        for b in (xd, wd, rd, y):
            b.free()
        L.free()


@pytest.mark.parametrize("gate,down,hidden,ff,n_experts,top_k,gemm", (
    (bm.Q4_K, bm.Q6_K, 2048, 768, 128, 8, 196),      # many experts of few slots
    (bm.Q6_K, bm.Q6_K, 2048, 768, 128, 8, 179),
    (bm.Q4_K, bm.Q6_K, 3072, 512, 256, 6, 410),
    (bm.Q6_K, bm.Q6_K, 7168, 2048, 1, 1, 73),        # one large expert: its tiles of 64 slots would leave the chip empty
    (bm.Q5_K, bm.Q6_K, 2048, 768, 8, 2, 56),
    (bm.Q4_K, bm.IQ4_XS, 4096, 1024, 24, 2, 79),
    (bm.IQ3_XXS, bm.IQ4_XS, 4096, 1024, 24, 2, 91),
    (bm.IQ2_XXS, bm.Q6_K, 2048, 768, 8, 3, 39),
    (bm.IQ2_XXS, bm.IQ2_XXS, 7168, 2048, 256, 8, 321),
    (bm.Q4_K, bm.Q6_K, 1024, 512, 256, 1, 3146),
))
def test_the_query_names_the_path_that_a_call_takes(gpu, gate, down, hidden, ff, n_experts, top_k, gemm):
    """bm_scratch_path_for, which is what a call asks, on both sides of the count from which the GEMM's launches are expected ahead, in
    both modes of the f32 order (the tolerance mode takes the GEMM from 96 tokens on at the latest: these gates have its kernels, but
    for IQ3_XXS), and where the caller has set a crossover of its own."""
    sc = gpu.scratch(gate, down, hidden, ff, n_experts, top_k, 4096)
    first = bm.PATH_PER_SLOT if hidden * ff < 1 << 23 or gate != bm.IQ2_XXS else bm.PATH_GROUPED
    try:
        for mode in (bm.GEMM_EXACT, bm.GEMM_FAST):
            gpu.set_gemm_mode(mode)
            early = mode == bm.GEMM_FAST and gemm > 96 and gate != bm.IQ3_XXS
            want = [first, bm.PATH_GROUPED, bm.PATH_GEMM if early else bm.PATH_GROUPED, bm.PATH_GEMM, bm.PATH_GEMM]
            assert [sc.path_for(m) for m in (21, 22, gemm - 1, gemm, 4096)] == want
            if early:
                assert [sc.path_for(m) for m in (95, 96)] == [bm.PATH_GROUPED, bm.PATH_GEMM]
        sc.set_path(bm.PATH_AUTO, 0, 4000)
        assert [sc.path_for(m) for m in (22, gemm, 3999, 4000)] == [bm.PATH_GROUPED, bm.PATH_GROUPED, bm.PATH_GROUPED, bm.PATH_GEMM]
    finally:
        gpu.set_gemm_mode(bm.GEMM_EXACT)
        sc.free()


@pytest.mark.parametrize("types,n_experts,top_k,tokens", (
    ((bm.Q3_K, bm.Q3_K, bm.Q4_K), 24, 4, (23, 24, 25)),           # four slots an expert
    ((bm.IQ4_XS, bm.IQ4_XS, bm.IQ4_XS), 13, 4, (24, 25, 26, 39)),  # eight
    ((bm.Q3_K, bm.Q3_K, bm.IQ3_XXS), 12, 3, (24, 31, 32)),         # the down stack's eight
    ((bm.IQ2_XXS, bm.IQ2_XXS, bm.Q6_K), 8, 3, (24, 31, 32)),       # twelve
    ((bm.IQ2_XXS, bm.IQ2_XXS, bm.Q6_K), 8, 3, (72, 73)),           # where the choice changes
    ((bm.Q5_K, bm.Q5_K, bm.Q6_K), 8, 2, (89, 90)),
    ((bm.Q4_K, bm.Q4_K, bm.IQ4_XS), 8, 4, (21, 22)),
    ((bm.Q6_K, bm.Q6_K, bm.Q6_K), 1, 1, (193, 194)),
))
def test_the_automatic_choice_gives_the_oracles_bits_where_it_changes(gpu, types, n_experts, top_k, tokens):
    hidden, ff, m = 512, 768, max(tokens)
    L = Layer(gpu, types, hidden, ff, n_experts, 5300)
    rng = np.random.default_rng(5301)
    x = normal_f32(rng, (m, hidden))
    ids, wts = route(rng, m, n_experts, top_k)
    want, _ = L.oracle(x, ids, wts, top_k)
    xd, sel, wd = gpu.upload(x, np.float32), gpu.upload(ids, np.uint32), gpu.upload(wts, np.float32)
    y = gpu.buffer(np.float32, m * hidden)
    sc = gpu.scratch(types[0], types[2], hidden, ff, n_experts, top_k, m)
    try:
        for n in tokens:
            y.fill_bytes(0xFF)
            gpu.enqueue_moe_forward(sc, L.dg, L.du, L.dd, xd, sel, wd, None, n, y)
            assert_f32(y.download()[:n * hidden], want.reshape(-1)[:n * hidden], f"{n} tokens")
    finally:
        sc.free()
        for b in (xd, sel, wd, y):
            b.free()
        L.free()


def test_the_automatic_choice_follows_the_crossovers(gpu):
    sc = gpu.scratch(bm.Q4_K, bm.Q6_K, 2048, 768, 128, 8, 4096)
    try:
        assert [sc.path_for(m) for m in (1, 21, 22, 195, 196, 4096)] == [bm.PATH_PER_SLOT, bm.PATH_PER_SLOT, bm.PATH_GROUPED,
                                                                       bm.PATH_GROUPED, bm.PATH_GEMM, bm.PATH_GEMM]
        gpu.set_gemm_mode(bm.GEMM_FAST)  # the tolerance mode's GEMM is faster: its cut comes earlier
        try:
            assert [sc.path_for(m) for m in (21, 22, 95, 96)] == [bm.PATH_PER_SLOT, bm.PATH_GROUPED, bm.PATH_GROUPED, bm.PATH_GEMM]
        finally:
            gpu.set_gemm_mode(bm.GEMM_EXACT)
        sc.set_path(bm.PATH_AUTO, 4, 2000)
        assert [sc.path_for(m) for m in (3, 4, 1999, 2000)] == [bm.PATH_PER_SLOT, bm.PATH_GROUPED, bm.PATH_GROUPED, bm.PATH_GEMM]
        sc.set_path(bm.PATH_PER_SLOT)
        assert sc.path_for(1024) == bm.PATH_PER_SLOT and sc.path_for(1025) == bm.PATH_GROUPED  # past the fused step's token limit
        assert sc.path_for(0) == bm.ESHAPE and sc.path_for(4097) == bm.ESHAPE
        with pytest.raises(bm.GpuError) as e:
            sc.set_path(7)
        assert "bm_scratch_set_path" in str(e.value)
    finally:
        sc.free()
    # a shape whose slot columns do not fit the per-slot step's LDS (64 slots of ff 2048) goes grouped from the first token (and by
    # the GEMM from three: 48 slots an expert)
    sc = gpu.scratch(bm.Q4_K, bm.Q6_K, 512, 2048, 4, 64, 8)
    try:
        assert [sc.path_for(m) for m in (1, 2, 3, 8)] == [bm.PATH_GROUPED, bm.PATH_GROUPED, bm.PATH_GEMM, bm.PATH_GEMM]
        sc.set_path(bm.PATH_PER_SLOT)
        assert sc.path_for(1) == bm.PATH_GROUPED
    finally:
        sc.free()
    # every type has a grouped GEMM: the same cut for a layer of the added types
    sc = gpu.scratch(bm.IQ4_XS, bm.Q3_K, 512, 256, 4, 2, 512)
    try:
        # (a gate/up stack on Q8_K columns, four experts: the exact GEMM is ahead from where the per-slot step ends)
        assert [sc.path_for(m) for m in (21, 22, 95, 96, 500)] == [bm.PATH_PER_SLOT] + 4 * [bm.PATH_GEMM]
        sc.set_path(bm.PATH_GEMM)
        assert sc.path_for(3) == bm.PATH_GEMM
    finally:
        sc.free()
    for call, word in ((lambda: gpu.scratch(bm.Q4_K, bm.Q6_K, 2048, 768, 128, 8, 5121), "40960"),
                       (lambda: gpu.scratch(bm.Q4_K, bm.Q6_K, 2000, 768, 128, 8, 16), "256"),
                       (lambda: gpu.scratch(bm.Q4_K, 99, 2048, 768, 128, 8, 16), "type")):
        with pytest.raises(bm.GpuError) as e:
            call()
        assert word in str(e.value) and "bm_scratch_create" in str(e.value)


def test_a_slot_without_an_expert_on_the_grouped_path_of_few_slots(gpu):
    """The grouped path with no more slots than experts and Q8_K columns on both sides (gate . up and down slot by slot, the
    slot-aware quantizer of h between them): a host-served slot and an id past the stack
    add nothing, the sums over the live slots are the oracle's, only the id past the stack raises; the scratch is poisoned first so
    that a stale row of h would show."""
    hidden, ff, n_experts, top_k, m = 512, 256, 16, 3, 3
    L = Layer(gpu, (bm.IQ2_XXS, bm.IQ2_XXS, bm.IQ4_XS), hidden, ff, n_experts, 5300)
    rng = np.random.default_rng(5301)
    x = normal_f32(rng, (m, hidden))
    wts = np.array([[0.5, 0.3, 0.2], [0.2, 0.5, 0.3], [0.1, 0.6, 0.3]], np.float32)
    xd, wd = gpu.upload(x, np.float32), gpu.upload(wts, np.float32)
    y = gpu.buffer(np.float32, m * hidden)
    sc = gpu.scratch(bm.IQ2_XXS, bm.IQ4_XS, hidden, ff, n_experts, top_k, 4)
    sc.set_path(bm.PATH_GROUPED)
    try:
        for ids, live, raises in ((np.array([[1, bm.HOST_SLOT, 3], [bm.HOST_SLOT, 0, bm.HOST_SLOT], [0, 2, 15]], np.uint32),
                                   ([(1, 0.5), (3, 0.2)], [(0, 0.5)], [(0, 0.1), (2, 0.6), (15, 0.3)]), False),
                                  (np.array([[1, 99, 3], [2, 0, 1], [0, 16, 2]], np.uint32),
                                   ([(1, 0.5), (3, 0.2)], [(2, 0.2), (0, 0.5), (1, 0.3)], [(0, 0.1), (2, 0.3)]), True)):
            want = np.concatenate([L.oracle(x[t:t + 1], np.array([[e for e, _ in live[t]]], np.uint32),
                                            np.array([[w for _, w in live[t]]], np.float32), len(live[t]))[0] for t in range(m)])
            sel = gpu.upload(ids, np.uint32)
            gpu.fault_clear()
            for rep in range(2):
                y.fill_bytes(0xFF)
                gpu.enqueue_moe_forward(sc, L.dg, L.du, L.dd, xd, sel, wd, None, m, y)
                assert_f32(y.download(), want, f"call {rep}")
            if raises:
                assert gpu.fault()[1] & (1 << bm.SITE_EXPERT_ID)
            else:
                assert gpu.fault() == (bm.FAULT_NONE, 0)
            sel.free()
        gpu.fault_clear()
    finally:
        sc.free()
        for b in (xd, wd, y):
            b.free()
        L.free()


def test_a_slot_without_an_expert_adds_nothing_on_every_path(gpu):
    """A host-served slot and an id past the stack: the token's sum is the oracle's over its live slots on each path, and
    the id past the stack raises ExpertId. With host-served slots only, no path raises anything (the GEMM path's route table
    does not list them and its SwiGLU quantizer leaves their columns alone, crates/gpu/src/gemm/swiglu.rs:96-140)."""
    L = Layer(gpu, (bm.Q4_K, bm.Q4_K, bm.Q6_K), 512, 256, 4, 5200)
    rng = np.random.default_rng(5201)
    m, top_k = 3, 3
    x = normal_f32(rng, (m, 512))
    ids = np.array([[1, bm.HOST_SLOT, 3], [2, 0, 1], [0, 9, 2]], np.uint32)
    wts = np.array([[0.5, 0.3, 0.2], [0.2, 0.5, 0.3], [0.1, 0.6, 0.3]], np.float32)
    want = np.concatenate([L.oracle(x[:1], np.array([[1, 3]], np.uint32), np.array([[0.5, 0.2]], np.float32), 2)[0],
                           L.oracle(x[1:2], ids[1:2], wts[1:2], 3)[0],
                           L.oracle(x[2:], np.array([[0, 2]], np.uint32), np.array([[0.1, 0.3]], np.float32), 2)[0]])
    xd, sel, wd = gpu.upload(x, np.float32), gpu.upload(ids, np.uint32), gpu.upload(wts, np.float32)
    y = gpu.buffer(np.float32, m * 512)
    sc = gpu.scratch(bm.Q4_K, bm.Q6_K, 512, 256, 4, top_k, 8)
    try:
        for path, name in PATHS:
            sc.set_path(path)
            gpu.fault_clear()
            y.fill_bytes(0xFF)
            gpu.enqueue_moe_forward(sc, L.dg, L.du, L.dd, xd, sel, wd, None, m, y)
            assert_f32(y.download(), want, name)
            assert gpu.fault()[1] & (1 << bm.SITE_EXPERT_ID)  # (the refused slot's NaN rows may raise the quantizer's site too)
        gpu.fault_clear()
        # host-served slots only: the same sums over the live slots, and no fault on any path
        ids_h = np.array([[1, bm.HOST_SLOT, 3], [bm.HOST_SLOT, 0, bm.HOST_SLOT], [0, 2, 1]], np.uint32)
        want_h = np.concatenate([L.oracle(x[:1], np.array([[1, 3]], np.uint32), np.array([[0.5, 0.2]], np.float32), 2)[0],
                                 L.oracle(x[1:2], np.array([[0]], np.uint32), np.array([[0.5]], np.float32), 1)[0],
                                 L.oracle(x[2:], ids_h[2:], wts[2:], 3)[0]])
        sel_h = gpu.upload(ids_h, np.uint32)
        for path, name in PATHS:
            sc.set_path(path)
            y.fill_bytes(0xFF)
            gpu.enqueue_moe_forward(sc, L.dg, L.du, L.dd, xd, sel_h, wd, None, m, y)
            assert_f32(y.download(), want_h, name + ", host-served slots")
            assert gpu.fault() == (bm.FAULT_NONE, 0), name
        sel_h.free()
    finally:
        sc.free()
        for b in (xd, sel, wd, y):
            b.free()
        L.free()
