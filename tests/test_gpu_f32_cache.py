"""GPU parity of the f32 cache (rvllm's own cache dtype, src/kv_storage.rs:
84-104 zeroes f32 K/V; src/cuda/kv_storage.rs:65-100 allocates the device
pool in f32): append, gather, copy and inspection bit-exact against the
oracle's f32 cache, paged decode against the oracle's float64 attention over
the same f32 cells, all through the C ABI."""
from __future__ import annotations

import sys

import numpy as np
import pytest
import torch

from oracle import oracle as orc
from rvllm_amd import workloads as W
from rvllm_amd._lib import RvkvError
from rvllm_amd.kv_storage import HipDecodePlan, HipGatherPlan, HipKvStorage
from tests.gpu_util import dev_u32

pytestmark = pytest.mark.gpu

F32 = torch.float32
# f32 cells and f32 arithmetic (scores, softmax, accumulation): the error
# against float64 stays far inside the f16 cache's 2e-3.
ATOL_F32 = 1e-4


@pytest.fixture(autouse=True)
def _announce(request):
    print(f"\n[gpu] {request.node.name}", flush=True)
    sys.stdout.flush()
    yield
    torch.cuda.synchronize()


def _bits(a: np.ndarray) -> np.ndarray:
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


def test_f32_kats(golden):
    """The reference's KATs at the reference's own cache dtype: the raw
    cache and the gather hold the written values exactly
    (src/kv_storage.rs:193-237)."""
    g = golden["reference_kats"]["round_trip_across_blocks"]
    st = HipKvStorage(1, 3, 2, 1, 2, dtype=F32)
    k = torch.tensor(g["k"], dtype=torch.float32).reshape(4, 1, 2).cuda()
    st.write_tokens(0, dev_u32(g["block_ids"]), dev_u32(g["offsets"]), k, k)
    raw = st.read_blocks(0, 0, dev_u32([0, 1, 2]))
    assert raw.dtype == F32
    assert raw.cpu().reshape(-1).tolist() == g["raw_cache"]
    plan = HipGatherPlan([(g["tables"][0], 3), (g["tables"][1], 1)])
    ok = torch.zeros(2 * 1 * 3 * 2, device="cuda")
    ov = torch.zeros_like(ok)
    st.gather(0, plan, ok, ov)
    got = ok.cpu().tolist()
    assert got == ov.cpu().tolist()
    assert got[:6] == g["gather_prefix_a"]
    assert got[6:8] == g["gather_prefix_b"]
    u = golden["reference_kats"]["untouched_slots"]
    st2 = HipKvStorage(1, 1, 4, 1, 2, dtype=F32)
    t = torch.tensor(u["k"], dtype=torch.float32).reshape(1, 1, 2).cuda()
    st2.write_tokens(0, dev_u32([0]), dev_u32([2]), t, t)
    ok = torch.zeros(8, device="cuda")
    st2.gather(0, HipGatherPlan([([0], 4)]), ok, torch.zeros_like(ok))
    assert ok.cpu().tolist() == u["gather"]


@pytest.mark.parametrize("nkv,hd,bs", [(5, 64, 16), (1, 256, 16), (3, 2, 2),
                                       (2, 12, 3), (8, 128, 32)])
def test_f32_append_gather_copy_bit_exact(nkv, hd, bs):
    rng = np.random.default_rng(hd + nkv)
    nb = 29
    st = HipKvStorage(2, nb, bs, nkv, hd, dtype=F32)
    ref = orc.KvCache(nb, bs, nkv, hd, orc.F32)
    slots = rng.permutation(nb * bs)[: nb * bs // 2]
    k = (rng.standard_normal((len(slots), nkv, hd)) * 100).astype(np.float32)
    v = rng.standard_normal((len(slots), nkv, hd)).astype(np.float32)
    k[0, 0, 0], v[0, 0, 0] = np.inf, -0.0
    k[1, 0, 0] = 1e-42  # an f32 subnormal: f32 rows are copied, never rounded
    st.write_tokens(1, dev_u32(slots // bs), dev_u32(slots % bs),
                    torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda())
    ref.write_tokens(slots // bs, slots % bs, k, v)
    # f16 source rows widen exactly (every f16 is an f32)
    s16 = rng.permutation(nb * bs)[:7]
    k16 = rng.standard_normal((7, nkv, hd)).astype(np.float16)
    k16[0, 0, 0] = np.float16(6e-8)  # an f16 subnormal
    st.write_tokens(1, dev_u32(s16 // bs), dev_u32(s16 % bs),
                    torch.from_numpy(k16).cuda(), torch.from_numpy(-k16).cuda())
    ref.write_tokens(s16 // bs, s16 % bs, k16.astype(np.float32),
                     (-k16).astype(np.float32))
    ids = dev_u32(np.arange(nb))
    assert np.array_equal(_bits(st.read_blocks(1, 0, ids).cpu().numpy()),
                          _bits(ref.k))
    assert np.array_equal(_bits(st.read_blocks(1, 1, ids).cpu().numpy()),
                          _bits(ref.v))
    assert st.read_blocks(0, 0, ids).eq(0).all()  # the other layer untouched
    # gather into f32 (bit for bit) through the padded plan, ragged lengths
    tabs = [rng.permutation(nb)[:5].tolist(), rng.permutation(nb)[:3].tolist()]
    plan = HipGatherPlan([(tabs[0], 5 * bs - 1), (tabs[1], 2 * bs + 1)])
    n = 2 * nkv * plan.ctx_len * hd
    ok = torch.empty(n, device="cuda")
    ov = torch.empty(n, device="cuda")
    st.gather(1, plan, ok, ov)
    wk, wv = ref.gather(plan.block_idx.cpu().numpy().view(np.uint32), 2,
                        plan.max_blocks, plan.ctx_len)
    assert np.array_equal(_bits(ok.cpu().numpy()), _bits(wk.reshape(-1)))
    assert np.array_equal(_bits(ov.cpu().numpy()), _bits(wv.reshape(-1)))
    with pytest.raises(RvkvError, match="an f32 cache gathers into F32 only"):
        st.gather(1, plan, ok.half(), ov.half())
    # checksums over the f32 bytes agree with the oracle's
    cs = st.block_checksums(1, 0, ids).cpu().numpy().view(np.uint64)
    assert np.array_equal(cs, ref.checksums(0, np.arange(nb)))
    cv = st.block_checksums(1, 1, ids).cpu().numpy().view(np.uint64)
    assert np.array_equal(cv, ref.checksums(1, np.arange(nb)))
    # copy-on-write: every layer, K and V, bit for bit
    src, dst = int(slots[0] // bs), int(slots[1] // bs)
    if src == dst:
        dst = (src + 1) % nb
    st.copy_blocks(dev_u32([src]), dev_u32([dst]))
    ref.copy_blocks([src], [dst])
    assert np.array_equal(_bits(st.read_blocks(1, 0, ids).cpu().numpy()),
                          _bits(ref.k))
    assert np.array_equal(_bits(st.read_blocks(1, 1, ids).cpu().numpy()),
                          _bits(ref.v))


def _f32_pool(bs, nkv, hd, lens, seed):
    cfg = W.Config("f32", 9, 1, nkv, nkv, hd, bs, len(lens))
    db = W.ragged_batch(cfg, lens, seed=seed, extra_blocks=3)
    st = HipKvStorage(1, db.num_blocks, bs, nkv, hd, dtype=F32)
    ref = orc.KvCache(db.num_blocks, bs, nkv, hd, orc.F32)
    rng = np.random.default_rng(seed)
    n = db.num_blocks * bs
    k = rng.standard_normal((n, nkv, hd)).astype(np.float32)
    v = rng.standard_normal((n, nkv, hd)).astype(np.float32)
    slots = np.arange(n)
    st.write_tokens(0, dev_u32(slots // bs), dev_u32(slots % bs),
                    torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda())
    ref.write_tokens(slots // bs, slots % bs, k, v)
    return db, st, ref


@pytest.mark.parametrize("G,hd", [(3, 64), (2, 128), (4, 256), (7, 32),
                                  (1, 64), (8, 128)])
def test_f32_decode_vs_oracle(G, hd):
    """Uniform and planned decode (windows, an empty sequence, sequences
    long enough to split) and the decode step (the append fused into the
    decode launch; f32 and f16 source rows) over an f32 cache, against
    float64 attention over the same cells."""
    bs, nkv = 16, 2
    lens = np.array([1, 17, 300, 2500, 64, 5], np.uint32)
    db, st, ref = _f32_pool(bs, nkv, hd, lens, seed=G * 7 + hd)
    H = G * nkv
    rng = np.random.default_rng(hd - G)
    qn = rng.standard_normal((len(lens), H, hd)).astype(np.float32)
    q = torch.from_numpy(qn).cuda()
    padded = db.padded_tables()
    tab = dev_u32(padded)
    tables = padded.reshape(-1)
    ctx = lens.copy()
    ctx[5] = 0  # an empty sequence: zero output
    for window in (0, 100):
        out = st.paged_decode(0, q, tab, dev_u32(ctx), int(ctx.max()),
                              window=window)
        want = orc.paged_decode_f64(ref, qn, tables, db.max_blocks, ctx,
                                    window=window)
        assert np.abs(out.cpu().numpy() - want).max() < ATOL_F32, window
        assert out[5].eq(0).all()
    plan = HipDecodePlan(st, ctx, H)
    out = st.paged_decode_planned(0, plan, q, tab, dev_u32(ctx))
    want = orc.paged_decode_f64(ref, qn, tables, db.max_blocks, ctx)
    assert np.abs(out.cpu().numpy() - want).max() < ATOL_F32
    # decode step: each sequence's new row lands at slot ctx-1, bit for bit,
    # and is attended to in the same call
    nk = rng.standard_normal((len(lens), nkv, hd)).astype(np.float32)
    nv = rng.standard_normal((len(lens), nkv, hd)).astype(np.float32)
    plan.update(lens)
    for use_plan in (False, True):
        got = st.decode_step(0, torch.from_numpy(nk).cuda(),
                             torch.from_numpy(nv).cuda(),
                             dev_u32(db.slot_block), dev_u32(db.slot_off), q,
                             tab, dev_u32(lens), int(lens.max()),
                             plan=plan if use_plan else None)
        want = orc.decode_step(ref, db.slot_block, db.slot_off, nk, nv,
                               tables, db.max_blocks, lens, qn)
        assert np.abs(got.cpu().numpy() - want).max() < ATOL_F32, use_plan
        ids = dev_u32(np.arange(db.num_blocks))
        assert np.array_equal(_bits(st.read_blocks(0, 0, ids).cpu().numpy()),
                              _bits(ref.k))
        assert np.array_equal(_bits(st.read_blocks(0, 1, ids).cpu().numpy()),
                              _bits(ref.v))
        nk, nv = nv, nk
    # f16 source rows: widened exactly into the f32 cells
    nk16 = rng.standard_normal((len(lens), nkv, hd)).astype(np.float16)
    nv16 = rng.standard_normal((len(lens), nkv, hd)).astype(np.float16)
    got = st.decode_step(0, torch.from_numpy(nk16).cuda(),
                         torch.from_numpy(nv16).cuda(), dev_u32(db.slot_block),
                         dev_u32(db.slot_off), q, tab, dev_u32(lens),
                         int(lens.max()), plan=plan)
    want = orc.decode_step(ref, db.slot_block, db.slot_off,
                           nk16.astype(np.float32), nv16.astype(np.float32),
                           tables, db.max_blocks, lens, qn)
    assert np.abs(got.cpu().numpy() - want).max() < ATOL_F32
    ids = dev_u32(np.arange(db.num_blocks))
    assert np.array_equal(_bits(st.read_blocks(0, 0, ids).cpu().numpy()),
                          _bits(ref.k))
    assert np.array_equal(_bits(st.read_blocks(0, 1, ids).cpu().numpy()),
                          _bits(ref.v))


def test_f32_smollm2_config():
    """configs[0] (SmolLM2-360M attention: 15 q heads over 5 KV heads,
    head_dim 64, 8 sequences with ctx in [17, 512]) at the reference's own
    cache dtype: the decode step against the oracle's restatement of
    rvllm's CPU path (write_tokens, padded gather, batch_mask and
    gqa_attention in f32, src/model.rs:628-644)."""
    db = W.smollm2_batch()
    c = db.cfg
    rng = W.Rng(c.seed)
    nb, bs = db.num_blocks, c.block_size
    st = HipKvStorage(1, nb, bs, c.n_kv_heads, c.head_dim, dtype=F32)
    ref = orc.KvCache(nb, bs, c.n_kv_heads, c.head_dim, orc.F32)
    slots = np.arange(nb * bs)
    k = rng.normal((nb * bs, c.n_kv_heads, c.head_dim))
    v = rng.normal((nb * bs, c.n_kv_heads, c.head_dim))
    st.write_tokens(0, dev_u32(slots // bs), dev_u32(slots % bs),
                    torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda())
    ref.write_tokens(slots // bs, slots % bs, k, v)
    nk = rng.normal((db.batch, c.n_kv_heads, c.head_dim))
    nv = rng.normal((db.batch, c.n_kv_heads, c.head_dim))
    q = rng.normal((db.batch, c.n_heads, c.head_dim))
    out = st.decode_step(0, torch.from_numpy(nk).cuda(),
                         torch.from_numpy(nv).cuda(), dev_u32(db.slot_block),
                         dev_u32(db.slot_off), torch.from_numpy(q).cuda(),
                         dev_u32(db.padded_tables()), dev_u32(db.ctx_lens),
                         int(db.ctx_lens.max()))
    want = orc.decode_step(ref, db.slot_block, db.slot_off, nk, nv,
                           db.padded_tables().reshape(-1), db.max_blocks,
                           db.ctx_lens, q)
    assert np.abs(out.cpu().numpy() - want).max() < ATOL_F32
    ids = dev_u32(np.arange(nb))
    assert np.array_equal(_bits(st.read_blocks(0, 1, ids).cpu().numpy()),
                          _bits(ref.v))




@pytest.mark.parametrize("G,hd,bs,Q,prior,window", [
    (3, 64, 16, 5, [0, 30], 0),          # less than one tile of rows or keys
    (3, 64, 16, 32, [1, 2000], 0),       # pieces beside a short prompt
    (1, 32, 4, 33, [0, 127, 96], 0),     # the smallest block, tile edges
    (4, 32, 8, 70, [900], 300),
    (2, 128, 16, 64, [64, 0], 0),
    (2, 128, 32, 21, [1700], 1000),
    (4, 256, 16, 40, [0, 700], 0),
    (1, 256, 128, 100, [3], 40),
    (5, 64, 16, 700, [0], 0),            # whole tiles seen by every row
])
def test_f32_prefill(G, hd, bs, Q, prior, window):
    """Prefill on the f32 matrix cores against float64, with ragged read
    counts, windows, cut keys and an out-of-range block id. Every product and
    sum is f32: 2e-5, as for the reference's own f32 cases."""
    from tests.test_gpu_parity import _prefill_f64
    rng = np.random.default_rng(hd + Q)
    nkv, prior = 2, np.asarray(prior)
    B, read = len(prior), prior + Q
    read[-1] = max(1, read[-1] - 2)
    mb = -(-int((prior + Q).max()) // bs)
    nb = B * mb + 3
    st = HipKvStorage(1, nb, bs, nkv, hd, dtype=torch.float32)
    at = torch.arange(nb * bs, device="cuda")
    k, v = (torch.randn(nb * bs, nkv, hd, device="cuda") for _ in range(2))
    st.write_tokens(0, (at // bs).int(), (at % bs).int(), k, v)
    tables = rng.permutation(nb)[:B * mb].reshape(B, mb).astype(np.uint32)
    q = torch.randn(B, Q, nkv * G, hd, device="cuda")
    for bad in (None, (int(read[0]) // 2) // bs):
        if bad is not None:
            tables[0, bad] = nb + 9
        t, p, r = dev_u32(tables), dev_u32(prior), dev_u32(read)
        out = st.paged_prefill(0, q, t, p, r, window=window)
        want = _prefill_f64(st, q, tables, prior, read, window)
        assert (out - want).abs().max() < 2e-5
        assert torch.equal(st.paged_prefill(0, q, t, p, r, window=window),
                           out)


@pytest.mark.parametrize("hd", [32, 64, 128, 256])
def test_f32_prefill_inf_value(hd):
    """A V row that is not finite reaches the rows that see it, and no
    others, wherever it lies in a key tile."""
    from tests.test_gpu_parity import _prefill_f64
    Q, nb, bs = 100, 7, 16
    table = np.random.default_rng(hd).permutation(nb).astype(np.uint32)
    for key in (0, 37, 63, 64, 99):
        st = HipKvStorage(1, nb, bs, 1, hd, dtype=torch.float32)
        k, v = (torch.randn(Q, 1, hd, device="cuda") for _ in range(2))
        at = np.arange(Q)
        slots = dev_u32(table[at // bs]), dev_u32(at % bs)
        st.write_tokens(0, *slots, k, v)
        q = torch.randn(1, Q, 2, hd, device="cuda")
        args = dev_u32(table[None]), dev_u32([0]), dev_u32([Q])
        want = _prefill_f64(st, q, table[None], [0], [Q], 0)
        v[key, 0, hd // 2] = float("inf")
        st.write_tokens(0, *slots, k, v)
        out = st.paged_prefill(0, q, *args)
        assert torch.isfinite(out[0, :key]).all()
        assert torch.isinf(out[0, key:, :, hd // 2]).all()
        out[0, key:, :, hd // 2] = want[0, key:, :, hd // 2].float()
        assert (out - want).abs().max() < 2e-5


@pytest.mark.parametrize("hd", [32, 64, 128, 256])
def test_f32_attn_prep_equals_f16_pool(hd):
    """attn_prep into an f32 pool: q bit for bit as on an f16 pool, whose
    cells are the f32 pool's rounded (one kernel, two cell types)."""
    rows, H, KV, nb = 37, 6, 2, 5
    g = torch.Generator("cuda").manual_seed(hd)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)
    qkv, bias = rnd(rows, (H + 2 * KV) * hd), rnd((H + 2 * KV) * hd)
    qn, kn, c, s = rnd(hd), rnd(hd), rnd(rows, hd // 2), rnd(rows, hd // 2)
    at = np.random.default_rng(hd).permutation(nb * 16)[:rows]
    out = []
    for dt in (torch.float32, torch.float16):
        st = HipKvStorage(1, nb, 16, KV, hd, dtype=dt)
        q = st.attn_prep_qkv(0, qkv, H, c, s, dev_u32(at // 16),
                             dev_u32(at % 16), bias=bias, q_norm=qn, k_norm=kn)
        ids = dev_u32(np.arange(nb))
        out.append([q] + [st.read_blocks(0, w, ids).half() for w in (0, 1)])
    for a, b in zip(*out):
        assert torch.equal(a, b)


def test_f32_prefill_block_past_32_bit_rows():
    """One block of 2^23 tokens at head_dim 256 (8 GiB of K, 8 of V): a row's
    byte offset in its block passes 2^32 from token 2^22 on. Rows and keys
    there against float64; every product and sum is f32: 2e-5."""
    bs, hd, Q, window = 1 << 23, 256, 40, 70
    p0 = (1 << 22) + 1000
    st = HipKvStorage(1, 1, bs, 1, hd, dtype=torch.float32)
    n = window + Q
    pos = np.arange(p0 - window, p0 + Q)
    k, v = (torch.randn(n, 1, hd, device="cuda") for _ in range(2))
    st.write_tokens(0, dev_u32(0 * pos), dev_u32(pos), k, v)
    q = torch.randn(1, Q, 2, hd, device="cuda")
    out = st.paged_prefill(0, q, dev_u32([[0]]), dev_u32([p0]),
                           dev_u32([p0 + Q]), window=window)
    j, i = torch.arange(n, device="cuda"), torch.arange(Q, device="cuda")
    see = (j[None] <= i[:, None] + window) & (j[None] > i[:, None])
    s = torch.einsum("qhd,kd->hqk", q[0].double(), k[:, 0].double())
    s = (s / hd ** 0.5).masked_fill(~see, -torch.inf)
    want = (torch.softmax(s, -1) @ v[:, 0].double()).transpose(0, 1)
    assert (out[0] - want).abs().max() < 2e-5


@pytest.mark.parametrize("hd", [32, 64, 128, 256])
@pytest.mark.parametrize("prior", [100, 1900])  # keys whole, and cut
def test_f32_prefill_inf_value_without_weight(hd, prior):
    """A V row that is not finite, behind a score so low that its weight is 0
    in f32 (2^-430 and less), stays out of every row: single keys anywhere in
    a key tile, and a run of them that fills a tile, which is all that some
    wave or piece has seen by then."""
    Q, bs = 40, 16
    n = prior + Q
    nb = -(-n // bs)
    table = np.random.default_rng(hd).permutation(nb).astype(np.uint32)
    at = np.arange(n)
    slots = dev_u32(table[at // bs]), dev_u32(at % bs)
    st = HipKvStorage(1, nb, bs, 1, hd, dtype=torch.float32)
    q = 1 + 0.1 * torch.randn(1, Q, 2, hd, device="cuda")
    for keys in ([0], [31], [64], [prior - 5], list(range(40)),
                 list(range(64, 96)), list(range(prior - 40, prior))):
        k, v = (torch.randn(n, 1, hd, device="cuda") for _ in range(2))
        k[keys] = -350 / hd ** 0.5  # (score ~ -350; the others within +-6)
        v[keys] = 0
        st.write_tokens(0, *slots, k, v)
        # (float64 weights of those keys are 1e-140: v = 0 there is the same)
        want = _prefill_f64_of(st, q, table, prior, n)
        v[keys, 0, 3] = float("inf")
        v[keys, 0, hd - 1] = float("nan")
        st.write_tokens(0, *slots, k, v)
        out = st.paged_prefill(0, q, dev_u32(table[None]), dev_u32([prior]),
                               dev_u32([n]))
        assert (out - want).abs().max() < 2e-5, keys[0]


def _prefill_f64_of(st, q, table, prior, n):
    from tests.test_gpu_parity import _prefill_f64
    return _prefill_f64(st, q, table[None], [prior], [n], 0)


def test_f32_prefill_position_near_2_32():
    """Positions up to 2^32 - 1 are past every key: a row there sees all of
    them (no wrap to position 0), cut keys or whole."""
    hd, bs, Q = 64, 16, 9
    for n in (200, 3000):
        nb = -(-n // bs)
        st = HipKvStorage(1, nb, bs, 1, hd, dtype=torch.float32)
        at = np.arange(n)
        k, v = (torch.randn(n, 1, hd, device="cuda") for _ in range(2))
        st.write_tokens(0, dev_u32(at // bs), dev_u32(at % bs), k, v)
        q = torch.randn(1, Q, 2, hd, device="cuda")
        t = dev_u32(np.arange(nb)[None])
        want = st.paged_prefill(0, q, t, dev_u32([n]), dev_u32([n]))
        for off in (2 ** 32 - 1, 2 ** 32 - 5, 2 ** 31):
            out = st.paged_prefill(0, q, t, dev_u32([off]), dev_u32([n]))
            assert torch.equal(out, want), off


@pytest.mark.parametrize("hd", [32, 64, 128, 256])
@pytest.mark.parametrize("batch", [128, 129])  # 256 workgroups, and more
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_f32_decode_step_appended_row(hd, batch, dtype):
    """The appended row loaded ahead of the keys and after them: the f32
    decode of the step and the row in the cache, against float64 (f32 products
    and sums: 2e-5)."""
    nkv, bs, mb = 2, 16, 6
    st = HipKvStorage(1, batch * mb, bs, nkv, hd, dtype=torch.float32)
    at = np.arange(batch * mb * bs)
    rnd = lambda *s: torch.randn(*s, device="cuda")
    st.write_tokens(0, dev_u32(at // bs), dev_u32(at % bs),
                    rnd(len(at), nkv, hd), rnd(len(at), nkv, hd))
    rng = np.random.default_rng(hd)
    tables = rng.permutation(batch * mb).reshape(batch, mb).astype(np.uint32)
    lens = rng.integers(1, mb * bs + 1, batch)
    lens[:3] = 1, 64, mb * bs
    pos = lens - 1
    k, v = (rnd(batch, nkv, hd).to(dtype) for _ in range(2))
    q = rnd(batch, nkv * 3, hd)
    blk = tables[np.arange(batch), pos // bs]
    out = st.decode_step(0, k, v, dev_u32(blk), dev_u32(pos % bs), q,
                         dev_u32(tables), dev_u32(lens), mb * bs)
    for w, x in ((0, k), (1, v)):
        got = st.read_blocks(0, w, dev_u32(blk))
        assert torch.equal(got[range(batch), pos % bs], x.float())
    from tests.test_gpu_parity import _prefill_f64
    want = _prefill_f64(st, q[:, None], tables, pos, lens, 0)
    assert (out - want[:, 0]).abs().max() < 2e-5


@pytest.mark.parametrize("hd", [64, 256])
def test_f32_prefill_cut_keys_streams_and_capture(hd):
    """Calls queued on three streams at once (the first two cut the keys, the
    third does not) and a captured one (not cut) replayed between them: each
    against float64 (f32 products and sums: 2e-5)."""
    Q, nkv, H, bs, prior = 40, 1, 4, 16, 3000
    n = prior + Q
    nb = -(-n // bs)
    table = np.random.default_rng(hd).permutation(nb).astype(np.uint32)
    at = np.arange(n)
    st = HipKvStorage(1, nb, bs, nkv, hd, dtype=torch.float32)
    st.write_tokens(0, dev_u32(table[at // bs]), dev_u32(at % bs),
                    *(torch.randn(n, nkv, hd, device="cuda")
                      for _ in range(2)))
    t, p, r = dev_u32(table[None]), dev_u32([prior]), dev_u32([n])
    qs = [torch.randn(1, Q, H, hd, device="cuda") for _ in range(4)]
    want = [_prefill_f64_of(st, q, table, prior, n) for q in qs]
    outs = [torch.empty_like(q) for q in qs]
    own, streams = st.stream, [torch.cuda.Stream() for _ in range(3)]
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        st.set_stream(torch.cuda.current_stream())
        st.paged_prefill(0, qs[3], t, p, r, out=outs[3])
    for _ in range(3):
        for o in outs:
            o.zero_()
        torch.cuda.synchronize()
        for q, o, s in zip(qs, outs, streams):
            st.set_stream(s)
            st.paged_prefill(0, q, t, p, r, out=o)
        graph.replay()
        torch.cuda.synchronize()
        for o, w in zip(outs, want):
            assert (o - w).abs().max() < 2e-5
    st.set_stream(own)
    assert torch.equal(*(st.paged_prefill(0, qs[0], t, p, r)
                         for _ in range(2)))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_whole_sequence_plan_with_appended_row(dtype):
    """A plan that keeps sequences whole past its item size (30 ragged ones to
    1500), with the step's rows appended: against float64, and the rows in the
    cache."""
    from rvllm_amd.kv_storage import HipDecodePlan
    from tests.test_gpu_parity import _prefill_f64
    nkv, G, hd, bs, batch, mb = 8, 2, 128, 16, 30, 94
    st = HipKvStorage(1, batch * mb, bs, nkv, hd, dtype=dtype)
    at = np.arange(batch * mb * bs)
    rnd = lambda *s: torch.randn(*s, device="cuda").to(dtype)
    st.write_tokens(0, dev_u32(at // bs), dev_u32(at % bs),
                    rnd(len(at), nkv, hd), rnd(len(at), nkv, hd))
    rng = np.random.default_rng(5)
    tables = rng.permutation(batch * mb).reshape(batch, mb).astype(np.uint32)
    lens = np.linspace(100, 1500, batch).astype(int)
    pos = lens - 1
    plan = HipDecodePlan(st, lens, nkv * G)
    if dtype == torch.float16:  # (an f32 row is twice the bytes)
        assert plan.items == batch
    k, v = (torch.randn(batch, nkv, hd, device="cuda") for _ in range(2))
    q = torch.randn(batch, nkv * G, hd, device="cuda")
    blk = tables[np.arange(batch), pos // bs]
    out = st.decode_step(0, k, v, dev_u32(blk), dev_u32(pos % bs), q,
                         dev_u32(tables), dev_u32(lens), plan=plan)
    for w, x in ((0, k), (1, v)):
        got = st.read_blocks(0, w, dev_u32(blk))[range(batch), pos % bs]
        assert torch.equal(got, x.to(dtype))
    want = _prefill_f64(st, q[:, None], tables, pos, lens, 0)
    # (f16: probabilities and packed products in f16, as every decode test)
    tol = 2e-5 if dtype == torch.float32 else 2e-3
    assert (out - want[:, 0]).abs().max() < tol


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("hd,G", [(128, 2), (64, 4), (256, 8)])
def test_decode_empty_batch(hd, G, dtype):
    """The size queries answer for an empty batch (no partials), and a decode
    of one returns at once."""
    st = HipKvStorage(1, 4, 16, 1, hd, dtype=dtype)
    for ctx in (0, 1, 5000):
        assert st.decode_partition_tokens(0, G, ctx) > 0
        assert st.decode_workspace_bytes(0, G, ctx) == 0
    none = torch.empty(0, dtype=torch.int32, device="cuda")
    out = st.paged_decode(0, torch.empty(0, G, hd, device="cuda"),
                          none.view(0, 4), none, 5000)
    assert out.shape == (0, G, hd)
