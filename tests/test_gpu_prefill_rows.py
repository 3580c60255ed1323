"""GPU parity of the row tiles' dispatch: whole-row K loads (one workgroup per
tile) and shares of a tile's blocks merged from the queue's buffer, against
the fragment-order kernel on the same pages (a plan with `waves` given), at
the sizes where they can go wrong: shares of unequal length, tiles too short
to split beside split ones, columns that see nothing of a share, every page
form, a rejected request, captures with and without a reservation, and
enqueues beside another queue's capture."""
import gc

import numpy as np
import pytest

from gpu_util import PrefillRunner, RaggedRunner, bf16_host, nan_bf16, to_dev_i32
from test_gpu_prefill_wide import assert_close

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def L():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import loom_infer_hip as L
    return L


# (hq, hkv, query rows, kv lengths, split)
CASES = [
    (32, 8, [1], [4111], True),                    # one share per 32 blocks
    (32, 8, [4, 3], [8200, 9], True),              # a one-block request beside a long one
    (8, 1, [5, 3, 2], [4099, 6001, 2050], True),   # group 8, unequal requests
    (32, 8, [40], [2065], True),                   # tiles ending inside the last share
    (28, 4, [9, 9], [2049, 2500], True),           # a group of 7 across tiles
    (8, 8, [1, 16], [2300, 2301], True),           # group 1
    (32, 8, [33, 64], [33, 250], False),           # short contexts
    (32, 8, [64, 65, 70], [700, 65, 900], False),  # many tiles of a request
    (32, 32, [24] * 4, [4100, 4096, 4097, 4111], False),  # many long streams
]


def case_inputs(case, form):
    import torch
    hq, hkv, qo_lens, kv_lens, _ = case
    P = 64 if "64" in form else 32 if "32" in form else 16
    rng = np.random.default_rng(sum(kv_lens) + P)
    pages = [(n + P - 1) // P for n in kv_lens]
    nnz, pool = sum(qo_lens), sum(pages) + 3
    ip = np.concatenate([[0], np.cumsum(pages)]).astype(np.int32)
    ix = rng.permutation(pool)[: ip[-1]].astype(np.int32)
    last = np.array([n - (p - 1) * P for n, p in zip(kv_lens, pages)], np.int32)
    qo = np.concatenate([[0], np.cumsum(qo_lens)]).astype(np.int32)
    g = torch.Generator(device="cuda").manual_seed(nnz)
    q = torch.randn(nnz * hq * 128, device="cuda", generator=g).to(torch.bfloat16)
    k, v = (torch.randn(pool * P * hkv * 128, device="cuda", generator=g) for _ in range(2))
    kw, scales = {"kv_page_size": P}, None
    if "hnd" in form:
        kw["kv_layout"] = "HND"
    if form.startswith("fp8"):
        kw["kv_dtype"] = "fp8_e4m3"
        scales = torch.tensor([0.8, 1.3], dtype=torch.float32, device="cuda")
        k, v = (x.to(torch.float8_e4m3fn).view(torch.uint8) for x in (k, v))
    else:
        k, v = k.to(torch.bfloat16), v.to(torch.bfloat16)
    return kw, pool, scales, [q, k, v], [qo, ip, ix, last]


def paged(L, case, kw, pool, scales, qkv, meta, **opts):
    import torch
    hq, hkv, qo_lens = case[:3]
    r = PrefillRunner(L, len(qo_lens), sum(qo_lens), pool, hq, hkv)
    r.spec = L.Bf16PagedPrefillSpec(len(qo_lens), sum(qo_lens), pool, hq, hkv, **kw)
    r.plan = r.provider.plan_bf16_paged(r.spec, **opts)
    assert r.plan.algorithm == "row_tile"
    held = r.queue.workspace_bytes
    out, lse = r.run_dev(*qkv, *(to_dev_i32(x) for x in meta), scales=scales)
    return (bf16_host(out), lse.view(torch.int32).cpu().numpy()), r.queue.workspace_bytes > held


@pytest.mark.parametrize("form", ["bf16", "bf16_hnd_page64", "fp8", "fp8_hnd_page32"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{c[1]}_{sum(c[2])}of{sum(c[3])}")
def test_planned_rows_match_the_fragment_order(L, oracle, case, form):
    kw, pool, scales, qkv, meta = case_inputs(case, form)
    here, scratch = paged(L, case, kw, pool, scales, qkv, meta)
    there, none = paged(L, case, kw, pool, scales, qkv, meta, waves=4)
    assert scratch == case[4] and not none
    assert not np.any(np.isnan(oracle.bf16_to_f32(here[0])))
    assert_close(oracle, [here, there])


def test_rejected_request_keeps_its_sentinels(L, oracle):
    case = CASES[2]
    kw, pool, scales, qkv, meta = case_inputs(case, "bf16")
    meta[2][meta[1][1] + 100] = pool  # a page of the second request out of range
    here, scratch = paged(L, case, kw, pool, scales, qkv, meta)
    there, _ = paged(L, case, kw, pool, scales, qkv, meta, waves=4)
    assert scratch
    rows = np.isnan(oracle.bf16_to_f32(here[0])).reshape(-1, 8 * 128).all(axis=1)
    assert list(np.nonzero(rows)[0]) == [5, 6, 7]
    assert_close(oracle, [here, there])


@pytest.mark.parametrize("case", CASES[:6], ids=lambda c: f"{c[0]}x{c[1]}_{sum(c[2])}of{sum(c[3])}")
def test_ragged_rows_match_the_fragment_order(L, oracle, case):
    import torch
    hq, hkv, qo_lens, kv_lens, _ = case
    qo = np.concatenate([[0], np.cumsum(qo_lens)]).astype(np.int32)
    kv = np.concatenate([[0], np.cumsum(kv_lens)]).astype(np.int32)
    nq, nkv = int(qo[-1]), int(kv[-1])
    g = torch.Generator(device="cuda").manual_seed(nkv)
    q, k, v = (torch.randn(n * h * 128, device="cuda", generator=g).to(torch.bfloat16)
               for n, h in ((nq, hq), (nkv, hkv), (nkv, hkv)))
    res = []
    for opts in ({}, {"waves": 4}):
        r = RaggedRunner(L, len(qo_lens), nq, nkv, hq, hkv, **opts)
        held = r.queue.workspace_bytes
        out, lse = r.run_dev(q, k, v, to_dev_i32(qo), to_dev_i32(kv))
        assert (r.queue.workspace_bytes > held) == (not opts)
        res.append((bf16_host(out), lse.view(torch.int32).cpu().numpy()))
    assert_close(oracle, res)


@pytest.mark.parametrize("reserved", [0, 1 << 24])
def test_captured_rows_replay(L, oracle, reserved):
    """A capture records the shares and their merge, with a reservation and
    without one (their states need none)."""
    import torch
    case = CASES[1]
    kw, pool, _, qkv, meta = case_inputs(case, "bf16")
    there, _ = paged(L, case, kw, pool, None, qkv, meta, waves=4)
    spec = L.Bf16PagedPrefillSpec(2, 7, pool, 32, 8, **kw)
    plan = L.PrefillProvider.load(0).plan_bf16_paged(spec)
    out = nan_bf16(spec.output_numel)
    lse = torch.full((spec.lse_numel,), float("nan"), dtype=torch.float32, device="cuda")
    dev = qkv + [to_dev_i32(x) for x in meta]
    q = L.GraphQueue(0, 2)
    if reserved:
        q.reserve_workspace(scratch_bytes=reserved)
    b = q.bindings(9)
    h = [b.bind_read(x) for x in dev]
    ho, hl = b.bind_read_write(out), b.bind_read_write(lse)
    args = L.Bf16PagedPrefillArgs(*h, ho.write(), hl.write())
    torch.cuda.synchronize()
    exec_ = q.capture(b, lambda scope: plan.enqueue_into(scope, args)).instantiate()
    for _ in range(3):
        out.fill_(float("nan"))
        lse.fill_(float("nan"))
        torch.cuda.synchronize()
        exec_.launch().wait()
        assert_close(oracle, [(bf16_host(out), lse.view(torch.int32).cpu().numpy()), there])
    exec_.into_bindings()


def shared_commands(L, oracle):
    """(plan, args of a binding set, capacity, outputs) of a row-tile prefill that
    runs in shares and of a single decode that runs as partitions."""
    import torch
    kw, pool, _, qkv, meta = case_inputs(CASES[1], "bf16")
    spec = L.Bf16PagedPrefillSpec(2, 7, pool, 32, 8, **kw)
    sspec = L.Bf16SingleDecodeSpec(4096, 32, 4)
    for plan, cls, dev, s in (
            (L.PrefillProvider.load(0).plan_bf16_paged(spec), L.Bf16PagedPrefillArgs,
             qkv + [to_dev_i32(x) for x in meta], spec),
            (L.DecodeProvider.load(0).plan_bf16(sspec), L.Bf16SingleDecodeArgs,
             [torch.randn(n * 128, device="cuda").to(torch.bfloat16)
              for n in (32, 4096 * 4, 4096 * 4)], sspec)):
        outs = (nan_bf16(s.output_numel),
                torch.full((s.lse_numel,), float("nan"), dtype=torch.float32, device="cuda"))

        def args(b, cls=cls, dev=dev, outs=outs):
            return cls(*[b.bind_read(x) for x in dev], *[b.bind_read_write(x).write() for x in outs])

        yield plan, args, len(dev) + 2, outs


def test_shared_commands_allocate_nothing(L, oracle):
    """The states of shared commands live in a buffer that the queue has from its
    creation on: the first enqueue on a fresh queue takes no device memory."""
    import torch
    for plan, args, n, outs in shared_commands(L, oracle):
        queues = [L.CommandQueue(torch.cuda.Stream(), 1) for _ in range(4)]
        gc.collect()  # (other tests' queues)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        for q in queues:
            b = q.bindings(n)
            a = args(b)
            scope = q.begin(b)
            plan.enqueue_into(scope, a)
            scope.finish().wait()
        assert torch.cuda.mem_get_info()[0] > free - (1 << 20)  # (each took 1 MiB or more)
        assert not any(torch.isnan(x).any() for x in outs)


def test_shared_commands_beside_a_capture(L, oracle):
    """While this thread captures a graph, an eager shared command on another,
    fresh queue runs and leaves the capture whole."""
    import torch
    cmds = list(shared_commands(L, oracle))
    for plan, args, n, outs in cmds:
        q = L.CommandQueue(torch.cuda.Stream(), 1)
        gq = L.GraphQueue(0, 1)
        torch.cuda.synchronize()
        b, gb = q.bindings(n), gq.bindings(n)
        held = [torch.empty_like(x) for x in outs]
        a, ga = args(b), args(gb, outs=held)
        pending = []

        def record(scope):
            plan.enqueue_into(scope, ga)
            eager = q.begin(b)
            plan.enqueue_into(eager, a)
            pending.append(eager.finish())

        graph = gq.capture(gb, record).instantiate()
        pending[0].wait()
        for _ in range(3):
            for x in held:
                x.fill_(float("nan"))
            torch.cuda.synchronize()
            graph.launch().wait()
            for x, y in zip(held, outs):
                assert torch.equal(x, y) and not torch.isnan(x).any()
        graph.into_bindings()


def test_shared_commands_in_a_callers_capture(L, oracle):
    """Captured by the caller into a graph of its own, whose replays the queue
    does not order, a command keeps off the queue's buffer and runs unshared,
    within the attention tolerance of the shared form."""
    import torch
    for plan, args, n, outs in shared_commands(L, oracle):
        stream = torch.cuda.Stream()
        eager, q = L.CommandQueue(stream, 1), L.CommandQueue(stream, 1)
        b = eager.bindings(n)
        a = args(b)
        torch.cuda.synchronize()
        scope = eager.begin(b)
        plan.enqueue_into(scope, a)
        scope.finish().wait()
        held = [torch.empty_like(x) for x in outs]
        b = q.bindings(n)
        a = args(b, outs=held)
        none = q.workspace_bytes
        scope = q.begin(b)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
            plan.enqueue_into(scope, a)
        scope.finish().wait()
        assert q.workspace_bytes == none < eager.workspace_bytes
        for _ in range(3):
            for x in held:
                x.fill_(float("nan"))
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert_close(oracle, [(bf16_host(o), l.view(torch.int32).cpu().numpy())
                                  for o, l in (held, outs)])


def test_rows_at_the_most_shares(L, oracle):
    """16 shares of each of 32 tiles fill the queue's buffer."""
    case = (32, 8, [16], [8209], True)
    kw, pool, scales, qkv, meta = case_inputs(case, "bf16")
    here, scratch = paged(L, case, kw, pool, scales, qkv, meta)
    there, _ = paged(L, case, kw, pool, scales, qkv, meta, waves=4)
    assert scratch
    assert_close(oracle, [here, there])
