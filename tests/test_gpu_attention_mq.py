"""GPU parity of the multi-query attention (the reference dispatch at
query_len > 1, attention_head256_f16kv.wgsl:72-267, and the decoder-layout
prefill entry point) against the CPU oracle: ora_attn_prefill on the f16
inputs for the causal case, and per query the oracle decode attention over
exactly the keys the reference's rules make visible (kv_start, sliding
window, softcap, non-causal).  Ring and paged caches are checked as storage
invariants: the same keys stored another way give the same output.
Contract: rel-L2 <= 1e-3."""
import numpy as np
import pytest

from doe_amd import DeviceBuffer, ops

pytestmark = pytest.mark.gpu

up = DeviceBuffer.from_array


def rel_l2(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def visible(abs_q, L, kv_start, causal, window):
    """Logical keys [lo, hi) of the query at abs_q (the reference's rule)."""
    hi = L
    if causal:
        hi = 0 if abs_q < kv_start else min(L, abs_q - kv_start + 1)
    lo = 0
    if window > 0 and abs_q >= window:
        mk = abs_q - window + 1
        if mk > kv_start:
            lo = min(L, mk - kv_start)
    return lo, hi


def oracle_rows(ora, q, k_rows, v_rows, hq, hkv, d, L, start_pos, kv_start, causal, window, scale, softcap):
    """Per query: the oracle decode attention over the visible cache rows
    (k_rows / v_rows: [capacity][hkv][d], logical key p at row kv_start + p)."""
    out = np.zeros((q.shape[0], hq, d), np.float32)
    for i in range(q.shape[0]):
        lo, hi = visible(start_pos + i, L, kv_start, causal, window)
        if hi <= lo:
            continue
        kr = np.ascontiguousarray(k_rows[kv_start + lo: kv_start + hi])
        vr = np.ascontiguousarray(v_rows[kv_start + lo: kv_start + hi])
        out[i] = ora.attn_decode(q[i], kr, vr, hq, hkv, d, hi - lo, hi - lo, scale, softcap=softcap, kv_layout=1)
    return out


@pytest.mark.parametrize("hq,hkv,d,ql,start", [(8, 4, 256, 37, 0), (8, 1, 512, 20, 5), (4, 4, 128, 100, 0),
                                               (16, 2, 64, 17, 30), (8, 8, 256, 16, 0), (2, 1, 512, 3, 0)])
def test_dispatch_causal_prompt_matches_oracle_prefill(dev, ora, hq, hkv, d, ql, start):
    # a prompt of ql queries at positions start .. start + ql - 1 over a cache
    # holding start + ql rows ([pos][kv_head][dim], the reference's order)
    print(f"[mq] hq={hq} hkv={hkv} d={d} ql={ql} start={start}", flush=True)
    rng = np.random.default_rng(hq * 100 + d + ql)
    L = start + ql
    cap = L + 3
    q = rng.standard_normal((ql, hq, d)).astype(np.float32)
    k = rng.standard_normal((cap, hkv, d)).astype(np.float16)
    v = rng.standard_normal((cap, hkv, d)).astype(np.float16)
    scale = 1.0 / np.sqrt(d)
    out = DeviceBuffer.empty((ql, hq, d), np.float32)
    ops.attention_dispatch(up(q), up(k), up(v), out, kv_capacity=cap, num_heads=hq, num_kv_heads=hkv, head_dim=d,
                           seq_len=L, query_len=ql, scale=scale, is_causal=1, start_pos=start)
    # ora_attn_prefill takes f32 K/V [kv_head][pos][dim]
    kf = np.ascontiguousarray(k[:L].astype(np.float32).transpose(1, 0, 2))
    vf = np.ascontiguousarray(v[:L].astype(np.float32).transpose(1, 0, 2))
    want = ora.attn_prefill(q, kf, vf, hq, hkv, d, ql, L, start, scale, True)
    err = rel_l2(out.download(), want)
    print(f"  rel_l2 {err:.2e}", flush=True)
    assert err <= 1e-3, err


@pytest.mark.parametrize("case", ["window", "softcap", "kv_start", "noncausal", "all_masked"])
def test_dispatch_key_rules_match_oracle(dev, ora, case):
    rng = np.random.default_rng(hash(case) % 1000)
    hq, hkv, d, ql = 8, 2, 256, 40
    cap = 96
    start, kv_start, causal, window, softcap, L = 30, 0, 1, 0, 0.0, 70
    if case == "window":
        window = 9
    elif case == "softcap":
        softcap = 0.5  # small cap: tanh saturates, the scores change visibly
    elif case == "kv_start":
        kv_start, start, L = 7, 40, 60  # logical key p at row 7 + p
    elif case == "noncausal":
        causal = 0
    else:  # queries before kv_start see nothing: zeros
        kv_start, start, L = 50, 0, 20
    q = (rng.standard_normal((ql, hq, d)) * 3).astype(np.float32)
    k = rng.standard_normal((cap, hkv, d)).astype(np.float16)
    v = rng.standard_normal((cap, hkv, d)).astype(np.float16)
    scale = 1.0 / np.sqrt(d)
    out = DeviceBuffer.empty((ql, hq, d), np.float32)
    ops.attention_dispatch(up(q), up(k), up(v), out, kv_capacity=cap, num_heads=hq, num_kv_heads=hkv, head_dim=d,
                           seq_len=L, query_len=ql, scale=scale, is_causal=causal, start_pos=start, kv_start=kv_start,
                           sliding_window=window, attn_softcap=softcap)
    want = oracle_rows(ora, q, k, v, hq, hkv, d, L, start, kv_start, causal, window, scale, softcap)
    got = out.download()
    if case == "all_masked":
        assert not want.any() and not got.any()
        return
    err = rel_l2(got, want)
    print(f"[mq {case}] rel_l2 {err:.2e}", flush=True)
    assert err <= 1e-3, err


def test_dispatch_ring_and_pages_are_storage_invariant(dev):
    # the same logical keys in a contiguous cache, a ring of `window` rows
    # (kv_layout 1) and pages (kv_layout 2) give the same prompt output
    rng = np.random.default_rng(77)
    hq, hkv, d, ql, start, window = 4, 2, 128, 24, 40, 16
    L = start + ql
    q = rng.standard_normal((ql, hq, d)).astype(np.float32)
    keys = rng.standard_normal((L, hkv, d)).astype(np.float16)
    vals = rng.standard_normal((L, hkv, d)).astype(np.float16)
    scale = 1.0 / np.sqrt(d)
    common = dict(num_heads=hq, num_kv_heads=hkv, head_dim=d, seq_len=L, query_len=ql, scale=scale, is_causal=1,
                  start_pos=start, sliding_window=window)
    o_flat = DeviceBuffer.empty((ql, hq, d), np.float32)
    ops.attention_dispatch(up(q), up(keys), up(vals), o_flat, kv_capacity=L, **common)
    # paged: page size 8, pages stored in reverse order
    ps = 8
    npg = (L + ps - 1) // ps
    table = np.arange(npg, dtype=np.uint32)[::-1].copy()
    kp = np.zeros((npg * ps, hkv, d), np.float16)
    vp = np.zeros_like(kp)
    for lp in range(npg):
        kp[table[lp] * ps: table[lp] * ps + ps][: min(ps, L - lp * ps)] = keys[lp * ps: lp * ps + ps]
        vp[table[lp] * ps: table[lp] * ps + ps][: min(ps, L - lp * ps)] = vals[lp * ps: lp * ps + ps]
    o_pg = DeviceBuffer.empty((ql, hq, d), np.float32)
    ops.attention_dispatch(up(q), up(kp), up(vp), o_pg, kv_capacity=npg * ps, page_table=up(table), kv_layout=2,
                           page_size=ps, **common)
    assert rel_l2(o_pg.download(), o_flat.download()) < 1e-6
    # ring: only the window's worth of rows exists; query i needs keys back to
    # start + i - window + 1, so a ring of `window` rows holds them only for
    # the last query -- check that query alone
    ring = np.zeros((window, hkv, d), np.float16)
    vring = np.zeros_like(ring)
    for p in range(L - window, L):
        ring[p % window] = keys[p]
        vring[p % window] = vals[p]
    # (query_len 1 runs the split-K decode kernel: the same query against the
    # flat cache through that kernel is the storage-invariant comparison; the
    # two kernels agree within the 1e-3 contract)
    o_ring = DeviceBuffer.empty((1, hq, d), np.float32)
    o_last = DeviceBuffer.empty((1, hq, d), np.float32)
    last = dict(common, query_len=1, start_pos=L - 1)
    ops.attention_dispatch(up(q[-1:]), up(ring), up(vring), o_ring, kv_capacity=window, kv_layout=1, **last)
    ops.attention_dispatch(up(q[-1:]), up(keys), up(vals), o_last, kv_capacity=L, **last)
    assert rel_l2(o_ring.download(), o_last.download()) < 1e-6
    assert rel_l2(o_last.download()[0], o_flat.download()[-1]) < 1e-3


@pytest.fixture
def mq_splits(request, dev):
    """Forces the multi-query attention's key split (attn_mq.splits; 0 the
    automatic choice, 1 none) and restores the automatic choice."""
    ops.tune("attn_mq.splits", request.param)
    yield request.param
    ops.tune("attn_mq.splits", 0)


@pytest.mark.parametrize("mq_splits", [0, 1, 2, 3, 5], indirect=True)
@pytest.mark.parametrize("hq,hkv,d", [(8, 4, 256), (4, 1, 512), (2, 1, 64)])
def test_prefill_f16kv_decoder_layout(dev, ora, hq, hkv, d, mq_splits):
    # the decoder's cache ([kv_head][max_seq][dim]) and the q part of fused
    # q/k/v rows (row stride q + 2 kv dims): a prompt continuing at position
    # 10, window 12, softcap 30; the key blocks split 1..5 ways over the grid
    # (5: more splits than key blocks, some empty) and merged
    rng = np.random.default_rng(d + hq)
    ql, start, maxs, window, softcap = 33, 10, 64, 12, 30.0
    L = start + ql
    row = (hq + 2 * hkv) * d
    qkv = rng.standard_normal((ql, row)).astype(np.float32)
    kc = rng.standard_normal((hkv, maxs, d)).astype(np.float16)
    vc = rng.standard_normal((hkv, maxs, d)).astype(np.float16)
    scale = 1.0 / np.sqrt(d)
    out = DeviceBuffer.empty((ql, hq * d + 8), np.float32)  # padded output rows
    ops.attention_prefill_f16kv(up(qkv), up(kc), up(vc), out, num_heads=hq, num_kv_heads=hkv, head_dim=d,
                                query_len=ql, kv_len=L, kv_stride=maxs, start_pos=start, scale=scale, softcap=softcap,
                                sliding_window=window, q_row_stride=row, out_row_stride=hq * d + 8)
    q = qkv[:, : hq * d].reshape(ql, hq, d)
    krows = np.ascontiguousarray(kc.transpose(1, 0, 2))
    vrows = np.ascontiguousarray(vc.transpose(1, 0, 2))
    want = oracle_rows(ora, q, krows, vrows, hq, hkv, d, L, start, 0, 1, window, scale, softcap)
    got = out.download()[:, : hq * d].reshape(ql, hq, d)
    err = rel_l2(got, want)
    print(f"[mq decoder layout {hq}/{hkv}x{d} splits {mq_splits}] rel_l2 {err:.2e}", flush=True)
    assert err <= 1e-3, err


@pytest.mark.parametrize("d,hq,hkv,ql,start,maxs,window,layout", [
    (64, 4, 2, 2, 0, 40, 0, 0), (64, 2, 2, 33, 97, 140, 0, 1), (64, 8, 1, 300, 0, 300, 50, 0),
    (128, 4, 4, 31, 1, 64, 0, 0), (128, 6, 3, 65, 300, 400, 128, 1), (128, 2, 1, 17, 3000, 3100, 0, 0),
    (256, 4, 2, 32, 0, 32, 0, 1), (256, 8, 4, 129, 31, 200, 33, 0), (256, 2, 1, 5, 2043, 2100, 0, 0),
    (256, 1, 1, 96, 0, 96, 1, 0)])
def test_prompt_blocks_against_float64(dev, d, hq, hkv, ql, start, maxs, window, layout):
    # around the edges of the 32-query and 32-key blocks, fewer blocks than
    # waves, windows that skip blocks, long caches (keys split over the grid);
    # cache rows past the prompt hold NaN (never written).  Bound: scores of
    # |s| < 8 from two f16 parts of Q (2^-22), P in two f16 parts (2^-22), f32
    # sums over kv keys (2^-24 sqrt(kv)).
    rng = np.random.default_rng(d + ql + start)
    kv = start + ql
    q = (rng.standard_normal((ql, hq, d)) * 10.0 ** rng.uniform(-2, 0.3, (ql, hq, 1))).astype(np.float32)
    k = np.full((hkv, maxs, d), np.nan, np.float16)
    v = np.full((hkv, maxs, d), np.nan, np.float16)
    k[:, :kv] = rng.standard_normal((hkv, kv, d))
    v[:, :kv] = rng.standard_normal((hkv, kv, d))
    scale = 1.0 / np.sqrt(d)
    out = DeviceBuffer.empty((ql, hq, d), np.float32)
    order = (0, 1, 2) if layout == 0 else (1, 0, 2)
    ops.attention_prefill_f16kv(up(q), up(k.transpose(order)), up(v.transpose(order)), out, num_heads=hq,
                                num_kv_heads=hkv, head_dim=d, query_len=ql, kv_len=kv, kv_stride=maxs,
                                start_pos=start, scale=scale, sliding_window=window, kv_layout=layout)
    got = out.download().astype(np.float64)
    pos, key = np.arange(start, kv)[:, None], np.arange(kv)[None, :]
    seen = (key <= pos) & ((key > pos - window) if window else True)
    for h in range(hq):
        g = h // (hq // hkv)
        s = q[:, h].astype(np.float64) @ k[g, :kv].astype(np.float64).T * scale
        s = np.where(seen, s, -np.inf)
        p = np.exp(s - s.max(1, keepdims=True))
        want = p @ v[g, :kv].astype(np.float64) / p.sum(1, keepdims=True)
        tol = 2.0 ** -22 * (8 + 1) + 2.0 ** -24 * np.sqrt(kv)
        assert rel_l2(got[:, h], want) <= tol, (h, rel_l2(got[:, h], want))


def float64_rows(q, k, v, key_rows, seen, scale, softcap=0.0):
    """softmax(q k^T) v in float64: q [ql][hq][d], caches [row][hkv][d], logical
    key p in row key_rows[p], seen [ql][keys]; also the largest |score|."""
    hq, hkv = q.shape[1], k.shape[1]
    out, top = np.zeros(q.shape), 0.0
    any_key = seen.any(1)
    for h in range(hq):
        g = h // (hq // hkv)
        s = q[:, h].astype(np.float64) @ k[key_rows, g].astype(np.float64).T * scale
        if softcap:
            s = np.tanh(s / softcap) * softcap
        top = max(top, np.abs(s[seen]).max(initial=0.0))
        s = np.where(seen, s, -np.inf)
        p = np.exp(s - np.where(any_key, s.max(1), 0.0)[:, None])
        out[:, h] = p @ v[key_rows, g].astype(np.float64) / np.where(any_key, p.sum(1), 1.0)[:, None]
    return out, top


def seen_keys(ql, keys, start, kv_start=0, window=0):
    pos, key = start + np.arange(ql)[:, None], np.arange(keys)[None, :] + kv_start
    return (key <= pos) & ((key > pos - window) if window else True)


def bound(queries, top, keys):
    # the 32-query form: Q in two f16 parts and f32 scores (2^-22 and a few
    # 2^-24 of the largest score), P in two f16 parts, f32 sums; the 16-query
    # form rounds P to one f16 (2^-11 of each term, at random)
    return 2.0 ** -22 * (top + 2) + 2.0 ** -24 * np.sqrt(keys) + (2.0 ** -11 if queries == 16 else 0.0)


@pytest.fixture
def mq_form(dev):
    def choose(splits, queries):
        ops.tune("attn_mq.splits", splits)
        ops.tune("attn_mq.queries", queries)
    yield choose
    choose(0, 0)


@pytest.mark.parametrize("queries", [0, 16])
@pytest.mark.parametrize("splits", [0, 1, 2, 3, 5, 16])
@pytest.mark.parametrize("d,hq,hkv,ql,start,window,softcap", [
    (64, 2, 1, 33, 10, 12, 30.0), (64, 4, 4, 40, 270, 0, 0.0), (128, 4, 2, 70, 300, 100, 0.0),
    (256, 8, 4, 33, 10, 12, 30.0), (256, 2, 1, 9, 700, 0, 5.0), (256, 4, 1, 64, 500, 260, 0.0)])
def test_key_splits_of_both_forms_against_float64(mq_form, d, hq, hkv, ql, start, window, softcap, splits, queries):
    # 1 to 16 key splits, some of them empty, with windows and softcaps
    rng = np.random.default_rng(d + ql + start)
    kv = start + ql
    q = rng.standard_normal((ql, hq, d)).astype(np.float32)
    k = rng.standard_normal((kv, hkv, d)).astype(np.float16)
    v = rng.standard_normal((kv, hkv, d)).astype(np.float16)
    scale = 1.0 / np.sqrt(d)
    out = DeviceBuffer.empty((ql, hq, d), np.float32)
    mq_form(splits, queries)
    ops.attention_prefill_f16kv(up(q), up(k), up(v), out, num_heads=hq, num_kv_heads=hkv, head_dim=d, query_len=ql,
                                kv_len=kv, kv_stride=kv, start_pos=start, scale=scale, softcap=softcap,
                                sliding_window=window, kv_layout=1)
    want, top = float64_rows(q, k, v, np.arange(kv), seen_keys(ql, kv, start, 0, window), scale, softcap)
    assert rel_l2(out.download(), want) <= bound(queries, top, kv)


@pytest.mark.parametrize("splits", [0, 3])
@pytest.mark.parametrize("layout,page", [(1, 0), (2, 16), (2, 7)])
@pytest.mark.parametrize("d,hq,hkv,ql,start,kv_start,window", [
    (64, 4, 2, 45, 200, 0, 130), (64, 2, 2, 2, 37, 3, 33), (128, 4, 1, 33, 90, 5, 64), (128, 2, 1, 100, 0, 0, 70),
    (256, 8, 4, 31, 300, 0, 257), (256, 2, 1, 65, 63, 11, 40)])
def test_ring_and_pages_of_several_queries(mq_form, d, hq, hkv, ql, start, kv_start, window, layout, page, splits):
    # key p in row (kv_start + p) % window of a ring, or through a page table
    # with the pages in any order; last key blocks partial, by three splits too,
    # with the key count from the host and from the device
    rng = np.random.default_rng(d + ql + start + page)
    L = start + ql - kv_start
    if layout == 1:
        cap, rows, extra = window, (kv_start + np.arange(L)) % window, {}
    else:
        npg = -(-(kv_start + L) // page) + 2
        cap, table = npg * page, rng.permutation(npg).astype(np.uint32)
        at = kv_start + np.arange(L)
        rows, extra = table[at // page].astype(np.int64) * page + at % page, {"page_table": up(table)}
    q = rng.standard_normal((ql, hq, d)).astype(np.float32)
    k = np.full((cap, hkv, d), np.nan, np.float16)  # rows that hold no key
    v = np.full((cap, hkv, d), np.nan, np.float16)
    k[rows] = rng.standard_normal((L, hkv, d))
    v[rows] = rng.standard_normal((L, hkv, d))
    scale = 1.0 / np.sqrt(d)
    want, top = float64_rows(q, k, v, rows, seen_keys(ql, L, start, kv_start, window), scale)
    mq_form(splits, 0)
    for source in (0, 1):
        out = DeviceBuffer.empty((ql, hq, d), np.float32)
        ops.attention_dispatch(up(q), up(k), up(v), out, kv_capacity=cap, kv_layout=layout, page_size=page,
                               num_heads=hq, num_kv_heads=hkv, head_dim=d, seq_len=L if source == 0 else 0,
                               kv_len_source=source, kv_len_buffer=up(np.array([L], np.uint32)) if source else None,
                               query_len=ql, scale=scale, is_causal=1, start_pos=start, kv_start=kv_start,
                               sliding_window=window, **extra)
        err = rel_l2(out.download(), want)
        assert err <= bound(0, top, L), (source, err)


def test_a_short_window_is_not_split_by_the_length_of_the_cache(mq_form):
    # 17 queries see 80 keys (four blocks) of 8000: one split by itself
    rng = np.random.default_rng(3)
    hq, hkv, d, ql, start, window = 8, 4, 256, 17, 7983, 64
    kv = start + ql
    q = rng.standard_normal((ql, hq, d)).astype(np.float32)
    k, v = up(rng.standard_normal((kv, hkv, d)).astype(np.float16)), up(rng.standard_normal((kv, hkv, d)).astype(np.float16))
    got = []
    for splits in (0, 1, 16):
        mq_form(splits, 0)
        out = DeviceBuffer.empty((ql, hq, d), np.float32)
        ops.attention_prefill_f16kv(up(q), k, v, out, num_heads=hq, num_kv_heads=hkv, head_dim=d, query_len=ql,
                                    kv_len=kv, kv_stride=kv, start_pos=start, scale=1 / 16, sliding_window=window,
                                    kv_layout=1)
        got.append(out.download())
    assert np.array_equal(got[0], got[1])
    assert rel_l2(got[2], got[1]) <= 2.0 ** -21


@pytest.mark.parametrize("layout,over", [(0, 0), (0, 1), (2, 0)])
def test_caches_about_two_gib(mq_form, layout, over):
    # the keys in the last rows of caches just under 2 GiB (the 32-query form,
    # 32-bit offsets) and just over (the 16-query form): the same bits as over
    # a cache of these rows alone
    rng = np.random.default_rng(5)
    hq, hkv, d, ql, L = 8, 8, 256, 40, 96
    cap = (1 << 31) // (hkv * d * 2) - (0 if over else 16)
    q = up(rng.standard_normal((ql, hq, d)).astype(np.float32))
    k = rng.standard_normal((L, hkv, d)).astype(np.float16)
    v = rng.standard_normal((L, hkv, d)).astype(np.float16)
    common = dict(num_heads=hq, num_kv_heads=hkv, head_dim=d, query_len=ql, scale=1 / 16, is_causal=1, seq_len=L)
    small = DeviceBuffer.empty((ql, hq, d), np.float32)
    mq_form(1, 16 if over else 0)
    ops.attention_dispatch(q, up(k), up(v), small, kv_capacity=L, start_pos=L - ql, **common)
    mq_form(1, 0)
    row = hkv * d * 2
    bk, bv = DeviceBuffer(cap * row), DeviceBuffer(cap * row)
    for buf, rows in ((bk, k), (bv, v)):
        buf.view((cap - L) * row, L * row).upload(rows)
    out = DeviceBuffer.empty((ql, hq, d), np.float32)
    if layout == 2:  # pages of 16 rows, the last six of the cache
        table = up(np.arange(cap // 16 - L // 16, cap // 16, dtype=np.uint32))
        ops.attention_dispatch(q, bk, bv, out, kv_capacity=cap, start_pos=L - ql, kv_layout=2, page_size=16,
                               page_table=table, **common)
    else:
        ops.attention_dispatch(q, bk, bv, out, kv_capacity=cap, start_pos=cap - ql, kv_start=cap - L, **common)
    assert np.array_equal(out.download(), small.download())


@pytest.mark.parametrize("d", [64, 128, 256, 512])
def test_query_rows_keep_to_themselves(dev, d):
    # a query of NaN, of an infinity, of zeros, of the largest values changes no
    # other query's bits; zeros see the mean of the values; a NaN query gives NaN
    # (head_dim 512's kernel: zeros, as for a query without keys)
    rng = np.random.default_rng(d)
    hq, hkv, ql = 2, 1, 40
    q = rng.standard_normal((ql, hq, d)).astype(np.float32)
    k = rng.standard_normal((ql, hkv, d)).astype(np.float16)
    v = rng.standard_normal((ql, hkv, d)).astype(np.float16)
    bad = q.copy()
    bad[3, 0, 5], bad[9, 1, 0], bad[17], bad[20], bad[35, :, :] = np.nan, np.inf, 0.0, 3e38, 1e-38
    outs = []
    for x in (q, bad):
        out = DeviceBuffer.empty((ql, hq, d), np.float32)
        ops.attention_prefill_f16kv(up(x), up(k), up(v), out, num_heads=hq, num_kv_heads=hkv, head_dim=d, query_len=ql,
                                    kv_len=ql, kv_stride=ql, start_pos=0, scale=0.1, kv_layout=1)
        outs.append(out.download())
    same = np.ones((ql, hq), bool)
    same[3, 0] = same[9, 1] = same[17] = same[20] = same[35] = False
    assert np.array_equal(outs[0][same], outs[1][same])
    assert np.isnan(outs[1][3, 0]).all() or d == 512
    mean = np.cumsum(v.astype(np.float64), 0) / np.arange(1, ql + 1)[:, None, None]
    for i in (17, 35):
        assert rel_l2(outs[1][i], np.broadcast_to(mean[i], (hq, d))) <= (1e-3 if d == 512 else 1e-6)
