"""GPU parity: the ragged multi-sequence batch (int8 MFMA BitLinear GEMMs,
per-token norms, attention of every token over its own sequence cache) vs
the oracle run token by token.

Reference semantics: multi_token_forward (src/model/multi_forward.rs:49-243)
with a pre-filled int8 KV cache, which is the sequential prefill of
src/model/generate.rs:151-160: every token of every sequence goes through
forward_with_cache in order.  Bar: every row of the batched BitLinear equals
the single-row SSE2-i8 path bit for bit; each sequence's last hidden, its
next greedy token and the new cache codes equal the oracle's bit for bit.
"""
import hashlib
import json
from pathlib import Path

import numpy as np
import pytest

import bitnet_synth as bs
import oracle.oracle as orc
import willamette_hip as wh
from oracle.oracle_model import OracleModel

pytestmark = pytest.mark.gpu


def bits_equal(a, b):
    a, b = np.asarray(a, np.float32), np.asarray(b, np.float32)
    return a.shape == b.shape and np.array_equal(a.view(np.uint32), b.view(np.uint32))


# --------------------------------------------------------------------------
# batched BitLinear (one GEMM over m token rows)
# --------------------------------------------------------------------------

# up to 512 output tiles of 64 x 64: the kernel whose waves split K; more
# (the last two): the kernel whose waves split the tokens
MATMUL_SHAPES = [(128, 64, 1), (256, 100, 5), (2560, 640, 16), (2560, 2560, 63), (2560, 2560, 64),
                 (2560, 2560, 65), (2560, 6912, 200), (6912, 2560, 37), (640, 65, 130),
                 (2560, 13824, 200), (1024, 13000, 150)]


@pytest.mark.parametrize("in_dim,out_dim,m", MATMUL_SHAPES)
def test_matmul_rows_equal_single_row_path(ctx, in_dim, out_dim, m):
    rng = np.random.default_rng(in_dim * 7 + out_dim * 3 + m)
    packed = rng.integers(0, 256, out_dim * in_dim // 4, dtype=np.uint8)
    scale = np.float32(rng.uniform(0.5, 2.0))
    x = rng.standard_normal((m, in_dim)).astype(np.float32) * np.float32(rng.uniform(0.1, 30))
    x[m // 2] = 0.0  # an all-zero row: scale 1, output exactly 0
    w = ctx.upload_i2s(packed, scale, in_dim, out_dim)
    y = wh.bitlinear_i2s_matmul_f32(ctx, w, x)
    for r in range(m):
        ry, _, _, _ = orc.bitlinear_i8(packed, scale, in_dim, out_dim, x[r])
        assert bits_equal(y[r], ry), f"row {r} of {m} differs from the SSE2-i8 path"
    w.close()


@pytest.mark.parametrize("in_dim,shift", [
    (128, 0), (1024, 0), (8192, 0),       # one unit of 16 columns per thread, the last a full workgroup
    (8320, 0), (16384, 0),                # two
    (16512, 0), (32768, 0),               # four
    (32896, 0),                           # more: the row read twice
    (2560, 1), (128, 3),                  # rows not 16-byte aligned
])
def test_matmul_quantiser_sizes(ctx, in_dim, shift):
    """The row quantiser at the row lengths and alignments where its kernels
    change, with NaN, infinite and zero rows: every output equals the
    single-row path's."""
    out_dim, m = 65, 5
    rng = np.random.default_rng(in_dim + shift)
    packed = rng.integers(0, 256, out_dim * in_dim // 4, dtype=np.uint8)
    x = (rng.standard_normal((m, in_dim)) * 3).astype(np.float32)
    x[1] = 0.0
    x[2, in_dim // 2] = np.nan
    x[3, in_dim - 1] = np.inf
    w = ctx.upload_i2s(packed, 0.75, in_dim, out_dim)
    dx = ctx.to_device(np.concatenate([np.zeros(shift, np.float32), x.ravel()]))
    dy = ctx.alloc(m * out_dim * 4)
    ctx.check(wh.lib.wm_bitlinear_i2s_matmul_f32_dev(ctx.h, w.h, dx.ptr + 4 * shift, m, dy.ptr))
    y = dy.to_host(np.float32).reshape(m, out_dim)
    for r in range(m):
        ry, _, _, _ = orc.bitlinear_i8(packed, np.float32(0.75), in_dim, out_dim, x[r])
        assert bits_equal(y[r], ry) or (np.isnan(ry).all() and np.isnan(y[r]).all()), f"row {r}"
    for b in (dx, dy, w):
        b.close()


def test_matmul_rejects_bad_lengths(ctx):
    rng = np.random.default_rng(5)
    w = ctx.upload_i2s(rng.integers(0, 256, 64 * 128 // 4, dtype=np.uint8), 1.0, 128, 64)
    x = np.zeros(3 * 128 + 1, np.float32)
    y = np.zeros(3 * 64, np.float32)
    with pytest.raises(wh.WillametteError) as e:
        ctx.check(wh.lib.wm_bitlinear_i2s_matmul_f32(ctx.h, w.h, wh._ptr(x, wh.C.c_float), x.size, 3,
                                                     wh._ptr(y, wh.C.c_float), y.size))
    assert e.value.kind == "Shape"
    w.close()


# --------------------------------------------------------------------------
# ragged batch forward
# --------------------------------------------------------------------------

SMALL = bs.BitNetConfig(n_layers=2, n_embd=256, n_ff=512, n_heads=2, n_kv_heads=1, head_dim=128,
                        vocab=1000, context_length=96)
GQA4 = bs.BitNetConfig(n_layers=3, n_embd=256, n_ff=384, n_heads=4, n_kv_heads=1, head_dim=64,
                       vocab=777, context_length=128)


@pytest.fixture(scope="module", params=[SMALL, GQA4], ids=["small", "gqa4"])
def pair(request, ctx):
    cfg = request.param
    hm = bs.make_host_model(cfg, seed=4321 + cfg.n_layers)
    dev = bs.load_device_model(ctx, hm)
    orm = OracleModel(hm)
    yield cfg, hm, dev, orm
    dev.close()
    orm.close()


def run_case(cfg, dev, orm, prefill, new_tokens, seed):
    """prefill[i] positions of N(0,1) K/V, then new_tokens[i] appended to
    sequence i in one batch; compared with the oracle token by token."""
    dkvs, okvs = [], []
    for i, n_pre in enumerate(prefill):
        dkv, okv = dev.kv_cache(cfg.context_length), orm.kv(cfg.context_length)
        if n_pre:
            k, v = bs.kv_prefill(cfg, seed=seed + i, n_pos=n_pre)
            dkv.append_positions(k, v)
            okv.append_positions(k, v)
        dkvs.append(dkv)
        okvs.append(okv)
    hidden, nxt = dev.batch_forward(dkvs, new_tokens)
    for i, toks in enumerate(new_tokens):
        okv = okvs[i]
        for tok in toks:
            rh = okv.forward(int(tok), okv.position)
        _, rnext = okv.logits_argmax(rh)
        assert bits_equal(hidden[i], rh), f"sequence {i}: last hidden differs"
        assert nxt[i] == rnext, f"sequence {i}: next token {nxt[i]} != {rnext}"
        assert dkvs[i].position == okv.position == prefill[i] + len(toks)
        n_pos = okv.position
        for l in range(cfg.n_layers):
            dk, dks, dv, dvs = dkvs[i].read_raw(l, n_pos)
            ok, oks, ov, ovs = okv.read_raw(l, n_pos)
            assert np.array_equal(dk, ok) and np.array_equal(dv, ov), f"seq {i} layer {l}: cache codes"
            assert bits_equal(dks, oks) and bits_equal(dvs, ovs), f"seq {i} layer {l}: cache scales"
    for kv in dkvs + okvs:
        kv.close()


def test_batch_single_sequence_from_empty_cache(pair):
    cfg, hm, dev, orm = pair
    run_case(cfg, dev, orm, [0], [[3, 17, 42, 7, 1]], seed=10)


def test_batch_ragged_sequences(pair):
    cfg, hm, dev, orm = pair
    rng = np.random.default_rng(cfg.n_layers)
    prefill = [0, 5, 40, 1, 63, 17]
    new = [[int(t) for t in rng.integers(0, cfg.vocab, n)] for n in (4, 1, 7, 2, 3, 1)]
    run_case(cfg, dev, orm, prefill, new, seed=20)


def test_batch_decode_step_all_single_tokens(pair):
    cfg, hm, dev, orm = pair
    rng = np.random.default_rng(7)
    prefill = [int(p) for p in rng.integers(1, cfg.context_length - 2, 9)]
    new = [[int(rng.integers(0, cfg.vocab))] for _ in prefill]
    run_case(cfg, dev, orm, prefill, new, seed=30)


DENSE = bs.BitNetConfig(n_layers=2, n_embd=256, n_ff=384, n_heads=2, n_kv_heads=1, head_dim=128,
                        vocab=500, context_length=4096)


def test_batch_dense_softmax_long_rows(ctx):
    """attn_q scaled down to 1e-6: every score is tiny and no softmax weight
    underflows, so each row's exact exp sum crosses many binades and runs
    over several 512-term steps with ragged tails (rows of 1 to ~3000
    positions), every tile live; ragged batch against the oracle token by
    token."""
    hm = bs.make_host_model(DENSE, seed=43)
    for hl in hm.layers:
        hl.scales["attn_q"] = 1e-6
    dev = bs.load_device_model(ctx, hm)
    orm = OracleModel(hm)
    rng = np.random.default_rng(12)
    prefill = [2999, 1030, 511, 0, 64]
    new = [[int(t) for t in rng.integers(0, DENSE.vocab, n)] for n in (3, 2, 4, 1, 6)]
    run_case(DENSE, dev, orm, prefill, new, seed=50)
    dev.close()
    orm.close()


# (head_dim, query heads per KV head, KV heads, context, new tokens, dense
# softmaxes, plan): rows' ends at 256, 512, 1024 and 2048 positions (the
# softmax's sizes), and what the plan chooses for the batch: tokens per work
# item of the scores, waves per row and float4s per lane of the softmax, query
# heads per wave of V
ATTENTION_CASES = [
    (64, 1, 4, 0, 3, True, (1, 1, 1, 1)),
    (64, 8, 1, 250, 9, True, (1, 1, 2, 1)),
    (64, 2, 2, 505, 11, True, (1, 1, 4, 1)),
    (128, 2, 1, 1020, 7, True, (1, 4, 2, 1)),
    (128, 8, 1, 2043, 8, False, (1, 4, 4, 1)),
    (128, 1, 4, 4064, 26, True, (2, 4, 4, 1)),    # the last tile reaches past the cache's 4090 positions
    (128, 4, 2, 63, 129, True, (1, 1, 1, 1)),
    (128, 4, 4, 0, 512, True, (2, 1, 2, 4)),
    (64, 4, 4, 1000, 300, False, (4, 1, 8, 1)),
    # heads that share a wave of V, the last workgroup's share ragged
    (64, 4, 4, 1000, 513, False, (8, 1, 8, 2)),
    (64, 4, 4, 900, 1025, True, (8, 1, 8, 4)),
    (128, 4, 4, 1500, 257, True, (8, 1, 8, 2)),
    (128, 8, 2, 700, 513, True, (4, 1, 8, 4)),
    # more than 2048 long dense rows: one wave each, two to four rounds of its sum
    (64, 4, 4, 1501, 151, True, (4, 1, 8, 1)),
    (64, 4, 4, 3001, 151, True, (8, 1, 16, 1)),
    # eight tokens per item of the scores, five in the last (with one query
    # head per KV head, not a multiple of the four rows of a step)
    (64, 1, 16, 3700, 29, True, (8, 4, 4, 1)),
    (64, 2, 16, 3700, 29, True, (8, 4, 4, 1)),
    (64, 8, 4, 3700, 109, True, (8, 1, 16, 1)),
    (128, 1, 16, 3500, 29, True, (8, 4, 4, 1)),
    (128, 2, 8, 3500, 61, True, (8, 4, 4, 1)),
]


@pytest.mark.parametrize("head_dim,group,n_kv,ctx_len,n_new,dense,plan", ATTENTION_CASES)
def test_batch_attention_sizes_match_decode(ctx, head_dim, group, n_kv, ctx_len, n_new, dense, plan):
    """One sequence's tokens in a batch against the same tokens decoded one at
    a time (checked against the oracle elsewhere): hidden state and cache
    bytes, the second layer's of every token among them."""
    n_embd = head_dim * group * n_kv
    assert tuple(wh.debug_batch_plan([ctx_len], [n_new], n_kv, group, head_dim).values()) == plan
    cfg = bs.BitNetConfig(n_layers=2, n_embd=n_embd, n_ff=384, n_heads=group * n_kv, n_kv_heads=n_kv,
                          head_dim=head_dim, vocab=300, context_length=4096)
    hm = bs.make_host_model(cfg, seed=head_dim + group)
    if dense:  # scores so small that no weight underflows
        for hl in hm.layers:
            hl.scales["attn_q"] = 1e-6
    dev = bs.load_device_model(ctx, hm)
    rng = np.random.default_rng(ctx_len + n_new)
    toks = rng.integers(0, cfg.vocab, n_new).tolist()
    a, b = dev.kv_cache(ctx_len + n_new), dev.kv_cache(ctx_len + n_new)
    if ctx_len:
        k, v = bs.kv_prefill(cfg, seed=9, n_pos=ctx_len)
        a.append_positions(k, v)
        b.append_positions(k, v)
    hidden, _ = dev.batch_forward([a], [toks])
    for t in toks:
        hb = b.forward(t, b.position)
    assert bits_equal(hidden[0], hb)
    for l in range(cfg.n_layers):
        assert all(np.array_equal(x, y) for x, y in zip(a.read_raw(l, a.position), b.read_raw(l, b.position)))
    a.close()
    b.close()
    dev.close()


@pytest.mark.parametrize("head_dim,group,n_kv,ctx_len,n_new,v_heads", [
    (64, 4, 4, 1000, 513, 2),
    (128, 4, 4, 1500, 257, 2),
    (64, 4, 4, 900, 1025, 4),
    (128, 8, 2, 700, 513, 4),
])
def test_batch_attention_heads_with_their_own_tiles(ctx, head_dim, group, n_kv, ctx_len, n_new, v_heads):
    """Softmaxes of a few positions each (queries of size ~400 against keys of
    unit size), so the heads that share a wave of V seldom share a live tile:
    the wave then takes them one after the other.  Against the same tokens
    decoded one at a time: hidden state and cache bytes."""
    assert wh.debug_batch_plan([ctx_len], [n_new], n_kv, group, head_dim)["v_heads"] == v_heads
    cfg = bs.BitNetConfig(n_layers=2, n_embd=head_dim * group * n_kv, n_ff=384, n_heads=group * n_kv,
                          n_kv_heads=n_kv, head_dim=head_dim, vocab=300, context_length=4096)
    hm = bs.make_host_model(cfg, seed=head_dim + n_new)
    for hl in hm.layers:
        hl.scales["attn_q"] *= 10.0
        hl.scales["attn_k"] = 1.0 / np.sqrt(cfg.n_embd * 2 / 3)
    dev = bs.load_device_model(ctx, hm)
    toks = np.random.default_rng(n_new).integers(0, cfg.vocab, n_new).tolist()
    a, b = dev.kv_cache(ctx_len + n_new), dev.kv_cache(ctx_len + n_new)
    k, v = bs.kv_prefill(cfg, seed=9, n_pos=ctx_len)
    a.append_positions(k, v)
    b.append_positions(k, v)
    hidden, _ = dev.batch_forward([a], [toks])
    for t in toks:
        hb = b.forward(t, b.position)
    assert bits_equal(hidden[0], hb)
    for l in range(cfg.n_layers):
        assert all(np.array_equal(x, y) for x, y in zip(a.read_raw(l, a.position), b.read_raw(l, b.position)))
    a.close()
    b.close()
    dev.close()


def test_batch_over_64_tokens(pair):
    # more than one 64-token GEMM tile, tiles shared by several sequences
    cfg, hm, dev, orm = pair
    rng = np.random.default_rng(11)
    prefill = [2, 0, 30]
    new = [[int(t) for t in rng.integers(0, cfg.vocab, n)] for n in (33, 29, 20)]
    run_case(cfg, dev, orm, prefill, new, seed=40)


def test_batch_rejects(pair):
    cfg, hm, dev, orm = pair
    a, b = dev.kv_cache(8), dev.kv_cache(8)
    for kvs, seqs in (([a, a], [[1], [2]]),            # the same cache twice
                      ([a, b], [[1], []]),             # an empty sequence
                      ([a], [[1] * 9]),                # past max_seq_len
                      ([a], [[cfg.vocab]])):           # token out of range
        with pytest.raises(wh.WillametteError):
            dev.batch_forward(kvs, seqs)
        assert a.position == 0 and b.position == 0
    a.close()
    b.close()


def test_batch_nonfinite_leaves_caches_untouched(ctx):
    cfg = SMALL
    hm = bs.make_host_model(cfg, seed=77)
    hm.layers[1].norms["ffn_sub_norm"][:] = np.inf
    dev = bs.load_device_model(ctx, hm)
    a, b = dev.kv_cache(cfg.context_length), dev.kv_cache(cfg.context_length)
    k, v = bs.kv_prefill(cfg, seed=3, n_pos=4)
    a.append_positions(k, v)
    with pytest.raises(wh.WillametteError) as e:
        dev.batch_forward([a, b], [[1, 2], [3]])
    assert e.value.kind == "NonFinite"
    assert a.position == 4 and b.position == 0
    a.close()
    b.close()
    dev.close()


def test_batch_bitnet2b_shape(ctx):
    """BitNet-2B shape: three sequences with contexts of 100, 1024 and 37
    pre-filled positions append 3, 1 and 2 tokens."""
    cfg = bs.BITNET_2B
    hm = bs.make_host_model(cfg, bs.master_seed(5))
    dev = bs.load_device_model(ctx, hm)
    orm = OracleModel(hm)
    try:
        run_case(cfg, dev, orm, [100, 1024, 37], [[15339, 11, 500], [128000], [7, 9]], seed=50)
    finally:
        dev.close()
        orm.close()


GOLDEN = Path(__file__).resolve().parent / "golden"


def test_batch_bitnet2b_ragged16_matches_oracle_fixture(ctx):
    """The benchmark's ragged step at its own size: BitNet-2B shape, 16
    sequences with contexts 1002-3842 appending 3-25 tokens each (257 in
    all), one wm_batch_forward.  Each sequence's next id, the SHA-256 of its
    last hidden and of its new cache rows must equal the oracle's
    token-by-token run recorded in tests/golden/bitnet2b_ragged16.json."""
    gold = json.loads((GOLDEN / "bitnet2b_ragged16.json").read_text())
    cfg = bs.BITNET_2B
    wl = bs.ragged_workload(cfg)
    assert [s["context"] for s in gold["sequences"]] == list(wl.contexts)
    hm = bs.make_host_model(cfg, bs.master_seed(4))
    dev = bs.load_device_model(ctx, hm)
    kvs = []
    for i, c in enumerate(wl.contexts):
        kv = dev.kv_cache(cfg.context_length)
        k, v = bs.kv_prefill(cfg, wl.prefill_seeds[i], c)
        kv.append_positions(k, v)
        del k, v
        kvs.append(kv)
    hidden, nxt = dev.batch_forward(kvs, wl.new_tokens)
    for i, rec in enumerate(gold["sequences"]):
        c, n = wl.contexts[i], len(wl.new_tokens[i])
        assert kvs[i].position == c + n
        assert nxt[i] == rec["next_id"], f"sequence {i}: next id"
        assert hashlib.sha256(np.ascontiguousarray(hidden[i], np.float32).tobytes()).hexdigest() == \
            rec["hidden_sha256"], f"sequence {i}: last hidden"
        h = hashlib.sha256()
        for layer in range(cfg.n_layers):
            k, ks, v, vs = kvs[i].read_raw(layer, c + n)
            for a in (k[c:], ks[c:], v[c:], vs[c:]):
                h.update(np.ascontiguousarray(a).tobytes())
        assert h.hexdigest() == rec["kv_sha256"], f"sequence {i}: new cache rows"
    for kv in kvs:
        kv.close()
    dev.close()
