"""GPU parity of the pipelined long-tile prefill kernels (32-token blocks in an
LDS ring, products and softmax of neighbouring blocks interleaved) at the
sizes where they can go wrong: remainders of the 64- and 128-column tiles,
causal ranges of one block and of several 64-block index windows, odd 16-row
block counts, wave groups with no block of their own, scores that move the
reference max, and every page form.  Against the oracle where it is quick and
against the 16-column algorithm on the same pages otherwise, within the
attention tolerance (gates/paged_batch_decode.rs:18-19: the weights are
rounded to BF16, at most 2^-9 each, far inside it)."""
import numpy as np
import pytest

from gpu_util import PrefillRunner, compare_decode, seeded_normal_bf16
from test_gpu_prefill import ragged_meta
from test_gpu_prefill_wide import assert_close, paged_pair

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def L():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import loom_infer_hip as L
    return L


# (hq, hkv, query rows, kv lengths): pools with room for long contexts, so the
# 64-column forms run pipelined
SMALL = [
    (32, 8, [1], [1]),                       # one token
    (32, 8, [16], [33]),                     # one tile, a second block of one token
    (32, 8, [17, 33], [1040, 2065]),         # index windows, odd blocks
    (28, 4, [19, 5], [300, 77]),             # a group of 7 across tiles
    (8, 8, [64, 65, 63], [64, 65, 1500]),    # group 1: tiles of 64 rows, whole prompts
    (8, 1, [9, 3, 40], [31, 32, 1056]),      # MQA
]


@pytest.mark.parametrize("shape", SMALL, ids=lambda s: f"{s[0]}x{s[1]}_{sum(s[2])}of{sum(s[3])}")
def test_small_grids_match_the_oracle(L, oracle, shape):
    hq, hkv, qo_lens, kv_lens = shape
    rng = np.random.default_rng(sum(kv_lens) + 77)
    pool = 2 * sum((n + 15) // 16 for n in kv_lens) + 2 * sum(qo_lens)
    qo, ip, ix, last = ragged_meta(rng, qo_lens, kv_lens, pool)
    B, nnz = len(qo_lens), int(qo[-1])
    q = seeded_normal_bf16(oracle, rng, nnz * hq * 128)
    k = seeded_normal_bf16(oracle, rng, pool * 16 * hkv * 128)
    v = seeded_normal_bf16(oracle, rng, pool * 16 * hkv * 128)
    ref = oracle.prefill(oracle.prefill_spec(B, nnz, pool, hq, hkv), q, k, v, qo, ip, ix, last)
    r = PrefillRunner(L, B, nnz, pool, hq, hkv, tile_cols="long")
    out, lse = r.run(q, k, v, qo, ip, ix, last)
    compare_decode(oracle, out, lse, *ref)


# (hq, hkv, rows, kv lengths, threads): the forms a plan takes by itself
PLANS = [
    (32, 8, [512], [1500], 512),                    # 64 columns, four groups
    (32, 8, [500, 90], [700, 2300], 256),           # 64 columns, two groups
    (32, 8, [2048], [2177], 512),                   # 128 columns, two groups
    (32, 8, [900, 1100, 1000], [900, 1100, 1900], 256),  # 128 columns, one group
]


@pytest.mark.parametrize("form", ["bf16", "bf16_hnd", "bf16_page64", "fp8", "fp8_hnd_page32"])
@pytest.mark.parametrize("plan", PLANS, ids=lambda s: f"{s[4]}t_{sum(s[2])}of{sum(s[3])}")
def test_planned_forms_match_row_tiles(L, oracle, plan, form):
    import torch
    hq, hkv, qo_lens, kv_lens, threads = plan
    P = 64 if "64" in form else 32 if "32" in form else 16
    rng = np.random.default_rng(sum(kv_lens) + P)
    pages = [(n + P - 1) // P for n in kv_lens]
    nnz, B = sum(qo_lens), len(qo_lens)
    pool = max(sum(pages) + 3, (2 * nnz + P - 1) // P)
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
        kw["kv_dtype"], scales = "fp8_e4m3", [0.8, 1.3]
        k, v = (x.to(torch.float8_e4m3fn).view(torch.uint8) for x in (k, v))
    else:
        k, v = k.to(torch.bfloat16), v.to(torch.bfloat16)
    p = L.PrefillProvider.load(0).plan_bf16_paged(
        L.Bf16PagedPrefillSpec(B, nnz, pool, hq, hkv, **kw))
    assert p.algorithm == "long_tile" and p.info.block_threads == threads
    res = paged_pair(L, B, nnz, pool, hq, hkv, q, k, v, qo, ip, ix, last, spec_kw=kw,
                     scales=scales, tile="long")
    assert not np.any(np.isnan(oracle.bf16_to_f32(res[0][0])))
    assert_close(oracle, res)


def test_growing_scores_move_the_reference_max(L, oracle):
    """Keys that grow along the context: the normalizer passes its refresh
    threshold again and again (scores rise by thousands in the log2 domain),
    early tokens' weights vanish, and the result stays the oracle's.  A score's
    FP32 rounding is up to 2^-24 of its magnitude (2^-9 here), so the LSE and
    the weights keep within the gate."""
    rng = np.random.default_rng(5)
    hq, hkv, rows, n = 16, 4, 40, 900
    pool = 200
    qo, ip, ix, last = ragged_meta(rng, [rows], [n], pool)
    q = np.abs(rng.standard_normal((rows, hq, 128), dtype=np.float32))
    k = rng.standard_normal((pool, 16, hkv, 128), dtype=np.float32)
    at = {int(p): i for i, p in enumerate(ix)}
    for p, i in at.items():
        for t in range(16):
            k[p, t] = np.abs(k[p, t]) * (16 * i + t) / 24.0
    qb, kb = oracle.bf16_from_f32(q.ravel()), oracle.bf16_from_f32(k.ravel())
    v = seeded_normal_bf16(oracle, rng, pool * 16 * hkv * 128)
    ref = oracle.prefill(oracle.prefill_spec(1, rows, pool, hq, hkv), qb, kb, v, qo, ip, ix, last)
    r = PrefillRunner(L, 1, rows, pool, hq, hkv, tile_cols="long")
    out, lse = r.run(qb, kb, v, qo, ip, ix, last)
    assert float(np.nanmax(np.abs(ref[1]))) > 500
    compare_decode(oracle, out, lse, *ref)


@pytest.mark.parametrize("batch", [65, 130])
def test_more_requests_than_a_wave(L, oracle, batch):
    """Batches past 64 requests take the workgroup-wide search for a tile."""
    rng = np.random.default_rng(batch)
    hq, hkv = 8, 2
    kv_lens = [int(x) for x in rng.integers(1, 70, size=batch)]
    qo_lens = [int(rng.integers(1, n + 1)) for n in kv_lens]
    pool = sum((n + 15) // 16 for n in kv_lens) + 2 * sum(qo_lens) // 16 + 3
    qo, ip, ix, last = ragged_meta(rng, qo_lens, kv_lens, pool)
    nnz = int(qo[-1])
    q = seeded_normal_bf16(oracle, rng, nnz * hq * 128)
    k = seeded_normal_bf16(oracle, rng, pool * 16 * hkv * 128)
    v = seeded_normal_bf16(oracle, rng, pool * 16 * hkv * 128)
    ref = oracle.prefill(oracle.prefill_spec(batch, nnz, pool, hq, hkv), q, k, v, qo, ip, ix, last)
    for tile in ("long", 16):
        r = PrefillRunner(L, batch, nnz, pool, hq, hkv, tile_cols=tile)
        out, lse = r.run(q, k, v, qo, ip, ix, last)
        compare_decode(oracle, out, lse, *ref)


# (hq, hkv, rows, kv lengths): ragged plans that run the pipelined tiles (64
# columns in four and two groups, 128 columns in two and one)
RAGGED = [
    (32, 8, [515], [515]),
    (32, 8, [300, 257], [1031, 300]),
    (32, 8, [2048], [2090]),
    (16, 2, [700, 513, 400], [700, 1300, 433]),
    (28, 4, [401, 999], [401, 1033]),
]


@pytest.mark.parametrize("shape", RAGGED, ids=lambda s: f"{s[0]}x{s[1]}_{sum(s[2])}of{sum(s[3])}")
def test_ragged_plans_match_row_tiles(L, oracle, shape):
    """The ragged contract's pipelined tiles keep 16 bits of every weight and
    FP32 normalizers, as its 16-column algorithm does: outputs differ by BF16
    rounding flips at most (one ulp of values below 4: 2^-6) and the LSE by
    FP32 summation order."""
    from gpu_util import RaggedRunner, bf16_host, to_dev_i32
    import torch
    hq, hkv, qo_lens, kv_lens = shape
    qo = np.concatenate([[0], np.cumsum(qo_lens)]).astype(np.int32)
    kv = np.concatenate([[0], np.cumsum(kv_lens)]).astype(np.int32)
    B, nq, nkv = len(qo_lens), int(qo[-1]), int(kv[-1])
    g = torch.Generator(device="cuda").manual_seed(nq)
    q, k, v = (torch.randn(n * h * 128, device="cuda", generator=g).to(torch.bfloat16)
               for n, h in ((nq, hq), (nkv, hkv), (nkv, hkv)))
    res = []
    for tile in (0, 16):
        r = RaggedRunner(L, B, nq, nkv, hq, hkv, tile_cols=tile)
        assert r.plan.algorithm == ("row_tile" if tile else "long_tile")
        out, lse = r.run_dev(q, k, v, to_dev_i32(qo), to_dev_i32(kv))
        res.append((oracle.bf16_to_f32(bf16_host(out)), lse.cpu().numpy()))
    (o, l), (eo, el) = res
    assert np.all(np.isfinite(o)) and np.abs(o - eo).max() <= 2.0 ** -6
    assert np.mean(o != eo) < 0.02
    assert np.abs(l - el).max() <= 1e-5


def pipe_and_rows(L, oracle, plan, form, make_k, v_scale=1.0):
    """((output, lse) of the plan's own algorithm, the 16-column algorithm's) on
    the same inputs, outputs divided by v_scale; |q| and keys from
    make_k(|normal|, token / kv_len)."""
    import torch
    from gpu_util import RaggedRunner, bf16_host, to_dev_i32
    hq, hkv, qo_lens, kv_lens = plan[:4]
    nnz, B = sum(qo_lens), len(qo_lens)
    g = torch.Generator(device="cuda").manual_seed(nnz)
    qo = np.concatenate([[0], np.cumsum(qo_lens)]).astype(np.int32)
    at = np.concatenate([np.arange(n) / n for n in kv_lens])
    n = len(at)
    q = torch.randn(nnz * hq * 128, device="cuda", generator=g).abs().to(torch.bfloat16)
    k, v = (torch.randn(n, hkv * 128, device="cuda", generator=g) for _ in range(2))
    k = make_k(k.abs(), torch.from_numpy(at).to("cuda", torch.float32)[:, None])
    # (below 4 one BF16 ulp, by which the rounding of the outputs may differ, is
    # the gate's 2^-6; the weights' rounding moves them by less)
    v = v.clamp(-3.75, 3.75) * v_scale
    res = []
    if form == "ragged":
        kv = np.concatenate([[0], np.cumsum(kv_lens)]).astype(np.int32)
        k, v = k.to(torch.bfloat16).flatten(), v.to(torch.bfloat16).flatten()
        for tile in (0, 16):
            r = RaggedRunner(L, B, nnz, n, hq, hkv, tile_cols=tile)
            assert r.plan.algorithm == ("row_tile" if tile else "long_tile")
            out, lse = r.run_dev(q, k, v, to_dev_i32(qo), to_dev_i32(kv))
            res.append((bf16_host(out), lse.view(torch.int32).cpu().numpy()))
    else:
        pages = [(x + 15) // 16 for x in kv_lens]
        pool = max(sum(pages) + 3, (2 * nnz + 15) // 16)
        ip = np.concatenate([[0], np.cumsum(pages)]).astype(np.int32)
        ix = np.random.default_rng(nnz).permutation(pool)[: ip[-1]].astype(np.int32)
        last = np.array([x - (p - 1) * 16 for x, p in zip(kv_lens, pages)], np.int32)
        row = np.concatenate([ix[ip[b] + np.arange(x) // 16].astype(np.int64) * 16 + np.arange(x) % 16
                              for b, x in enumerate(kv_lens)])
        pooled = []
        for x in (k, v):
            p = torch.zeros(pool * 16, hkv * 128, device="cuda")
            p[torch.from_numpy(row).cuda()] = x
            pooled.append(p.flatten())
        kw, scales = {}, None
        if form == "fp8":
            kw, scales = {"kv_dtype": "fp8_e4m3"}, [0.8, 0.9]
            k, v = (x.clamp(-440, 440).to(torch.float8_e4m3fn).view(torch.uint8) for x in pooled)
        else:
            k, v = (x.to(torch.bfloat16) for x in pooled)
        p = L.PrefillProvider.load(0).plan_bf16_paged(
            L.Bf16PagedPrefillSpec(B, nnz, pool, hq, hkv, **kw))
        assert p.algorithm == "long_tile" and p.info.block_threads == plan[4]
        res = paged_pair(L, B, nnz, pool, hq, hkv, q, k, v, qo, ip, ix, last, spec_kw=kw,
                         scales=scales, tile="long")
    # (powers of two: exact)
    return [(oracle.bf16_from_f32(oracle.bf16_to_f32(o) / np.float32(v_scale)), l) for o, l in res]


RANGE = [(p, "bf16") for p in PLANS] + [(p, "ragged") for p in RAGGED[:4]]


@pytest.mark.parametrize("plan,form", RANGE + [(p, "fp8") for p in PLANS],
                         ids=lambda x: x if isinstance(x, str) else f"{x[0]}x{x[1]}_{sum(x[2])}of{sum(x[3])}")
def test_references_that_move_again_and_again(L, oracle, plan, form):
    """Scores that rise by hundreds in the log2 domain along every context: each
    form rescales O and the normalizers every few blocks."""
    res = pipe_and_rows(L, oracle, plan, form, lambda k, at: k * at * 40)
    assert float(np.nanmax(np.abs(res[1][1].view(np.float32)))) > 300
    assert_close(oracle, res)


@pytest.mark.parametrize("exponent", [115, -120])
@pytest.mark.parametrize("plan,form", RANGE,
                         ids=lambda x: x if isinstance(x, str) else f"{x[0]}x{x[1]}_{sum(x[2])}of{sum(x[3])}")
def test_values_of_extreme_magnitude(L, oracle, plan, form, exponent):
    """V of about 2^115 and 2^-120 under scores that rise by some 20 in the log2
    domain: a weight is at most 1, so no sum of them with V leaves FP32's range
    unless the result does, and small products keep BF16's precision."""
    res = pipe_and_rows(L, oracle, plan, form, lambda k, at: k * at * 2, 2.0 ** exponent)
    assert_close(oracle, res)


@pytest.mark.parametrize("plan,form", RANGE,
                         ids=lambda x: x if isinstance(x, str) else f"{x[0]}x{x[1]}_{sum(x[2])}of{sum(x[3])}")
def test_runs_of_tokens_that_score_minus_infinity(L, oracle, plan, form):
    """Whole blocks of keys whose scores overflow to -inf, the context's second
    block among them, weigh nothing in every wave group."""
    def keys(k, at):
        k = k * 0.1
        r = ((at > 0.07) & (at < 0.21)) | ((at > 0.4) & (at < 0.45))
        return k.masked_fill(r, -3.0e38)
    assert_close(oracle, pipe_and_rows(L, oracle, plan, form, keys))


def ragged_pair(L, hq, hkv, qo, kv, q, k, v):
    """The long tiles' raw output bits and the 16-column algorithm's."""
    import torch
    from gpu_util import RaggedRunner, bf16_host, to_dev_i32
    res = []
    for tile in (0, 16):
        r = RaggedRunner(L, len(qo) - 1, int(q.numel()) // (hq * 128), int(k.numel()) // (hkv * 128),
                         hq, hkv, tile_cols=tile)
        assert r.plan.algorithm == ("row_tile" if tile else "long_tile")
        out, lse = r.run_dev(q, k, v, to_dev_i32(qo), to_dev_i32(kv))
        res.append((bf16_host(out), lse.view(torch.int32).cpu().numpy()))
    return res


# (hq, hkv, qo_indptr, kv_indptr): ranges that overlap an earlier request's (the
# later one owns the rest of its rows: tiles that do not begin at its first row),
# one that ends before it begins, and requests with fewer keys than rows, whose
# rows keep their sentinels; 64 and 128 columns
GUARDED = [
    (32, 8, [0, 400, 300, 700, 900], [0, 500, 600, 1300, 1400]),
    (32, 8, [0, 900, 610, 1700, 2300], [0, 900, 1000, 2400, 2900]),
    (28, 4, [0, 333, 1000, 777, 2100, 3000], [0, 433, 1100, 1200, 2800, 2900]),
]


@pytest.mark.parametrize("case", GUARDED, ids=lambda c: f"{c[0]}x{c[1]}_{c[2][-1]}")
def test_ragged_rows_go_to_their_owners(L, oracle, case):
    import torch
    hq, hkv, qo, kv = case
    g = torch.Generator(device="cuda").manual_seed(qo[-1])
    q, k, v = (torch.randn(n * h * 128, device="cuda", generator=g).to(torch.bfloat16)
               for n, h in ((qo[-1], hq), (kv[-1], hkv), (kv[-1], hkv)))
    res = ragged_pair(L, hq, hkv, np.int32(qo), np.int32(kv), q, k, v)
    dropped = np.isnan(oracle.bf16_to_f32(res[0][0])).reshape(qo[-1], -1)
    rows = np.zeros(qo[-1], bool)
    end = 0
    for s0, s1, p0, p1 in zip(qo, qo[1:], kv, kv[1:]):
        if s1 > max(s0, end) and not 0 < s1 - s0 <= p1 - p0:
            rows[max(s0, end):s1] = True
        end = max(end, s1)
    assert rows.any() and np.array_equal(dropped.all(axis=1), rows)
    assert_close(oracle, res)


@pytest.mark.parametrize("hq,hkv,batch,most", [(64, 8, 70, 40), (64, 8, 130, 120)])
def test_ragged_batches_past_a_wave(L, oracle, hq, hkv, batch, most):
    """More than 64 requests: the workgroup-wide search, with a request past its
    keys and one that overlaps the one before it."""
    import torch
    rng = np.random.default_rng(batch)
    rows = rng.integers(most // 2 + 14, most + 14, size=batch)
    kv = np.concatenate([[0], np.cumsum(rows + rng.integers(0, 9, size=batch))]).astype(np.int32)
    qo = np.concatenate([[0], np.cumsum(rows)]).astype(np.int32)
    kv[67:] -= rows[66]              # request 66: fewer keys than rows
    qo[33] += 7                      # request 32 takes the first rows of 33
    kv[33:] += 7
    g = torch.Generator(device="cuda").manual_seed(batch)
    q, k, v = (torch.randn(int(n) * h * 128, device="cuda", generator=g).to(torch.bfloat16)
               for n, h in ((qo[-1], hq), (kv[-1], hkv), (kv[-1], hkv)))
    res = ragged_pair(L, hq, hkv, qo, kv, q, k, v)
    dropped = np.isnan(oracle.bf16_to_f32(res[0][0])).reshape(int(qo[-1]), -1).all(axis=1)
    assert np.array_equal(np.nonzero(dropped)[0], np.arange(qo[66], qo[67]))
    assert_close(oracle, res)


def shifted(t, n):
    """A copy of `t` that begins n elements into its allocation."""
    import torch
    x = torch.empty(t.numel() + n, dtype=t.dtype, device=t.device)
    x[n:] = t
    return x[n:]


@pytest.mark.parametrize("form", ["bf16", "fp8", "ragged"])
@pytest.mark.parametrize("rows", [600, 2500])
def test_operands_on_four_byte_boundaries(L, oracle, rows, form):
    """Q, K, V and O four bytes past a 16-byte boundary give the bits of the
    aligned call: the tiles' loads straight into LDS and their row stores need no
    more than four."""
    import torch
    from gpu_util import RaggedRunner, bf16_host, nan_bf16, to_dev_i32
    hq, hkv, n = 32, 8, rows + 70
    g = torch.Generator(device="cuda").manual_seed(rows)
    q, k, v = (torch.randn(m * h * 128, device="cuda", generator=g)
               for m, h in ((rows, hq), (n + 26, hkv), (n + 26, hkv)))
    q = q.to(torch.bfloat16)
    by = 2
    if form == "fp8":
        k, v = (x[: (n + 26) // 16 * 16 * hkv * 128].to(torch.float8_e4m3fn).view(torch.uint8)
                for x in (k, v))
        by = 4
    else:
        k, v = k.to(torch.bfloat16), v.to(torch.bfloat16)
    got = []
    for move in (lambda x, m: x, shifted):
        out = move(nan_bf16(rows * hq * 128), 2)
        if form == "ragged":
            r = RaggedRunner(L, 1, rows, n + 26, hq, hkv)
            assert r.plan.algorithm == "long_tile"
            o, l = r.run_dev(move(q, 2), move(k, by), move(v, by), to_dev_i32([0, rows]),
                             to_dev_i32([0, n + 26]), out=out)
        else:
            pool = (n + 26) // 16
            used = (n + 15) // 16
            kk, vv = (x[: pool * 16 * hkv * 128] for x in (k, v))
            r = PrefillRunner(L, 1, rows, pool, hq, hkv)
            r.spec = L.Bf16PagedPrefillSpec(1, rows, pool, hq, hkv,
                                            kv_dtype="fp8_e4m3" if form == "fp8" else "bf16")
            r.plan = r.provider.plan_bf16_paged(r.spec)
            assert r.plan.algorithm == "long_tile"
            o, l = r.run_dev(move(q, 2), move(kk, by), move(vv, by), to_dev_i32([0, rows]),
                             to_dev_i32([0, used]), to_dev_i32(np.arange(used)[::-1]),
                             to_dev_i32([n - (used - 1) * 16]), out=out,
                             scales=torch.tensor([0.8, 0.9], device="cuda") if form == "fp8" else None)
        got.append((bf16_host(o.clone()), l.cpu().numpy()))
    assert not np.any(np.isnan(oracle.bf16_to_f32(got[0][0])))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])


@pytest.mark.parametrize("value", [float("inf"), float("nan")], ids=["inf", "nan"])
@pytest.mark.parametrize("plan,form", [(PLANS[0], "bf16"), (PLANS[3], "bf16"), (RAGGED[1], "ragged")],
                         ids=["four_groups", "one_group", "ragged"])
def test_infinite_and_nan_keys_stay_with_the_rows_that_see_them(L, oracle, plan, form, value):
    """A key that is infinite or not a number in the last rows of each context
    makes the rows that see it NaN, as in the 16-column algorithm, and leaves
    every earlier row alone (a masked score is replaced whatever it was)."""
    hq, hkv, qo_lens, kv_lens = plan[:4]

    def keys(k, at):
        n = np.repeat(kv_lens, kv_lens)
        import torch
        late = at[:, 0] * torch.from_numpy(n).to("cuda") > torch.from_numpy(n).to("cuda") - 20.5
        return k.masked_fill(late[:, None], value)

    res = pipe_and_rows(L, oracle, plan, form, keys)
    bad = np.isnan(oracle.bf16_to_f32(res[0][0])).reshape(sum(qo_lens), -1)
    want = np.concatenate([np.arange(r) >= r - 20 for r in qo_lens])
    assert np.array_equal(bad.all(axis=1), want) and np.array_equal(bad.any(axis=1), want)
    rows = np.repeat(~want, hq * 128)
    (o, l), (eo, el) = res
    assert_close(oracle, [(o[rows], l[np.repeat(~want, hq)]), (eo[rows], el[np.repeat(~want, hq)])])
