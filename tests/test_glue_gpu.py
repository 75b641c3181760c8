"""The glue ops of a decode step through their own C-ABI entry points, each against the CPU oracle
or a closed form: embedding gather, RMSNorm (with and without the residual add), dense GEMM at
every row-tile regime, fused classifier arg-max, row arg-max with ties, rotary tables, and the
q/k/v split + rotation + KV-cache store for head dimensions 32 and 64."""
import numpy as np
import pytest
import torch

from conftest import TOL_MAX, TOL_MEAN, rel_errors

pytestmark = pytest.mark.gpu


def test_embedding_lookup(ops):
    g = torch.Generator().manual_seed(1)
    V, H = 1000, 2880
    table = torch.randn(V, H, generator=g).to(torch.bfloat16)
    ids = torch.tensor([0, 999, 5, 5, 123, -3, 4000], dtype=torch.int32)        # out of range: clamped
    got = ops.embedding_lookup(table.cuda(), ids.cuda()).cpu()
    want = table.float()[ids.clamp(0, V - 1).long()]
    assert torch.equal(got, want)


@pytest.mark.parametrize("B,H", [(1, 256), (7, 2880), (300, 2880), (5, 5000), (3, 100)])
def test_rmsnorm_matches_oracle(ops, orc, B, H):
    rng = np.random.default_rng(B + H)
    x = rng.standard_normal((B, H)).astype(np.float32) * 3
    r = rng.standard_normal((B, H)).astype(np.float32)
    w = (1 + 0.1 * rng.standard_normal(H)).astype(np.float32)
    for residual in (None, r):
        xd = torch.from_numpy(x.copy()).cuda()
        t = ops.rmsnorm(xd, torch.from_numpy(w).cuda(), None if residual is None else torch.from_numpy(r).cuda())
        xin = x if residual is None else x + r
        assert np.array_equal(xd.cpu().numpy(), xin)                            # x += residual, in place
        want = np.stack([orc.rmsnorm(xin[b], w) for b in range(B)])
        want_bf16 = torch.from_numpy(want).to(torch.bfloat16).float().numpy()
        got = t.float().cpu().numpy()
        # the CPU arithmetic restated (double sum, float rsqrt): equal up to one bf16 rounding step
        assert np.abs(got - want_bf16).max() <= 2.0 ** -7 * np.abs(want).max()
        assert (got == want_bf16).mean() > 0.999


@pytest.mark.parametrize("B,N,K,bias", [(1, 64, 64, True), (33, 5120, 2880, True), (130, 2880, 4096, True),
                                        (600, 2880, 4096, True), (1024, 5120, 2880, False),
                                        (700, 4096, 256, True), (2304, 1056, 512, True)])
def test_dense_gemm(ops, B, N, K, bias):
    """Every regime of the dispatch: row tiles of 32..160 rows or 256 by estimated time, ragged last row tile and last column
    tile.  (The 256-row kernel by itself: test_tall_dense_gpu.py.)"""
    g = torch.Generator(device="cuda").manual_seed(B + N)
    a = torch.randn(B, K, device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda", generator=g) * 0.05).to(torch.bfloat16)
    b = (torch.randn(N, device="cuda", generator=g)).to(torch.bfloat16).float() if bias else None
    got = ops.dense_gemm(a, ops.pack_weight(w), N, b).cpu().numpy()
    want = (a.double() @ w.double().T + (b.double() if bias else 0)).cpu().numpy()
    assert np.abs(got - want).max() <= 2e-5 * np.abs(want).max() + 1e-6 * np.sqrt(K)


@pytest.mark.parametrize("B,N,K", [(2500, 2880, 4096), (2049, 5120, 2880), (4096, 288, 256)])
def test_dense_gemm_of_a_prompt_pass_equals_the_same_rows_in_small_batches(ops, B, N, K):
    """Thousands of rows, where most products run the kernel with 256-row tiles and both operands through LDS (here all but the
    narrow one): same bits per row as the streaming kernels, which run the batches of a fifth of the rows."""
    g = torch.Generator(device="cuda").manual_seed(B + N)
    a = torch.randn(B, K, device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, device="cuda", generator=g) * 0.05).to(torch.bfloat16)
    b = (torch.randn(N, device="cuda", generator=g)).to(torch.bfloat16).float()
    wp = ops.pack_weight(w)
    full = ops.dense_gemm(a, wp, N, b)
    step = B // 5 + 1
    for r0 in range(0, B, step):
        assert torch.equal(full[r0:r0 + step], ops.dense_gemm(a[r0:r0 + step].contiguous(), wp, N, b)), r0


# Tiles of 256 rows per XCD, 32 of which are a round: 12 (halves only), 74 (two rounds and halves; of the last tile's 52 rows, 33
# and 1, whose second half is 20, 1 and 0), 83 (two rounds, the rest whole)
@pytest.mark.parametrize("B,N,K", [(2048, 2880, 4096), (2100, 16640, 256), (2081, 16640, 256), (2049, 16640, 256), (2369, 16672, 320)])
def test_halves_of_the_tiles_in_a_last_round(ops, B, N, K):
    test_dense_gemm_of_a_prompt_pass_equals_the_same_rows_in_small_batches(ops, B, N, K)


@pytest.mark.parametrize("B,V,K", [(5, 4096, 256), (130, 201088, 2880), (1024, 50304, 512), (515, 9984, 256),
                                   (256, 9984, 512), (255, 4128, 320)])
def test_classifier_argmax_equals_argmax_of_logits(ops, B, V, K):
    g = torch.Generator(device="cuda").manual_seed(V)
    a = torch.randn(B, K, device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn(V, K, device="cuda", generator=g) * 0.05).to(torch.bfloat16)
    w[V - 1] = w[7]                                   # the same logit in the first and in the last, partly filled tile
    wp = ops.pack_weight(w)
    logits = ops.dense_gemm(a, wp, V)
    ids = ops.classifier_argmax(a, wp, V).cpu().numpy()
    assert np.array_equal(ids, logits.cpu().numpy().argmax(axis=1))
    assert np.array_equal(ops.argmax(logits).cpu().numpy(), ids)


@pytest.mark.parametrize("B", [130, 600])
@pytest.mark.parametrize("cols", [(7, 11, 40, 135, 300, 4127), (11, 40, 135), (135, 300), (200, 250), (259, 263)])
def test_classifier_argmax_ties_pick_the_lowest_column(ops, B, cols):
    """Equal maxima in the two half-waves of a lane pair, in two column blocks of a wave, in the two
    waves that share a row, in two column tiles and in the last, partly filled tile: the lowest
    column wins (run.cpp:739-750), on the streaming kernel (130 rows) and the 256-row kernel (600)."""
    V, K = 4128, 256
    g = torch.Generator(device="cuda").manual_seed(B)
    a = torch.randn(B, K, device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn(V, K, device="cuda", generator=g) * 0.05).to(torch.bfloat16)
    big = (w[cols[0]].float() * 8).to(torch.bfloat16)
    for c in cols:
        w[c] = big
    ids = ops.classifier_argmax(a, ops.pack_weight(w), V).cpu().numpy()
    logits = (a.float() @ w.float().T).cpu().numpy()
    wins = logits[:, cols[0]] >= logits.max(axis=1)               # rows where the repeated column is the maximum
    assert wins.sum() > B // 10
    assert (ids[wins] == min(cols)).all()


def test_argmax_ties_lowest_index(ops):
    x = np.full((4, 4096), -1.0, np.float32)
    x[0, [4095, 17, 2000]] = 3.0
    x[1, :] = 0.0
    x[2, 4095] = 1.0
    x[3, :] = -np.inf
    assert ops.argmax(torch.from_numpy(x).cuda()).cpu().tolist() == [17, 0, 4095, 0]


def test_rope_tables_match_oracle(ops, orc, synth):
    for cfg in (synth.tiny_config(2048), synth.gptoss20b_config(1024)):
        cs, sn = ops.rope_tables(cfg, 300)
        ocs, osn = orc.rope_tables(cfg, 300)
        assert np.array_equal(cs, ocs) and np.array_equal(sn, osn)


@pytest.mark.parametrize("D,n_q,n_kv", [(32, 8, 2), (64, 64, 8)])
def test_rope_kv_store_then_attention(ops, orc, synth, D, n_q, n_kv):
    """Positions are fed one by one through the rotation + store op, every sequence at its own
    position; q must be the half-split rotation of run.cpp:480-499 and attention over the cache the
    op filled must be the oracle's attention over the rotated keys and the values."""
    import dataclasses
    cfg = dataclasses.replace(synth.tiny_config(2048), head_dim=D, n_attn_heads=n_q, n_kv_heads=n_kv)
    B, S, cap = 3, 70, 128
    lens_final = np.array([70, 33, 1], np.int32)
    rng = np.random.default_rng(D)
    qkv_dim = (n_q + 2 * n_kv) * D
    qkv = rng.standard_normal((S, B, qkv_dim)).astype(np.float32)
    cs, sn = orc.rope_tables(cfg, S)
    cs_d, sn_d = torch.from_numpy(cs).cuda(), torch.from_numpy(sn).cuda()

    def rot(x, pos):                                  # x [..., D]
        h = D // 2
        x1, x2 = x[..., :h], x[..., h:]
        return np.concatenate([x1 * cs[pos] - x2 * sn[pos], x2 * cs[pos] + x1 * sn[pos]], -1)

    cache = ops.KVCache(B, n_kv, D, cap)
    cache.kv.view(torch.int16).fill_(0x7FC1)
    K = np.zeros((B, S, n_kv, D), np.float32)
    V = np.zeros((B, S, n_kv, D), np.float32)
    q_last = np.zeros((B, n_q, D), np.float32)
    for step in range(S):
        pos = np.minimum(step, lens_final - 1)        # a finished sequence rewrites its last position
        lens = torch.from_numpy((pos + 1).astype(np.int32)).cuda()
        q = ops.rope_kv_store(torch.from_numpy(qkv[step]).cuda(), cache, cs_d, sn_d, lens, n_q).cpu().numpy()
        for b in range(B):
            row = qkv[step, b]
            want_q = rot(row[: n_q * D].reshape(n_q, D), pos[b])
            np.testing.assert_allclose(q[b], want_q, rtol=1e-6, atol=1e-6)
            K[b, pos[b]] = rot(row[n_q * D:(n_q + n_kv) * D].reshape(n_kv, D), pos[b])
            V[b, pos[b]] = row[(n_q + n_kv) * D:].reshape(n_kv, D)
            q_last[b] = want_q
    bf = lambda a: torch.from_numpy(a).to(torch.bfloat16).float().numpy()
    sinks = rng.standard_normal(n_q).astype(np.float32)
    attn = ops.AttnDecode(B, n_q, n_kv, D, S)
    got = attn.forward(torch.from_numpy(q_last).cuda(), cache, torch.from_numpy(lens_final).cuda(),
                       torch.from_numpy(sinks).cuda()).float().cpu().numpy()
    want = orc.attn_decode(q_last, bf(K), bf(V), lens_final, sinks, 0)
    assert np.isfinite(got).all()
    mx, mean = rel_errors(got, want)
    assert mx <= TOL_MAX and mean <= TOL_MEAN, (mx, mean)


def test_rope_kv_store_skips_empty_sequences(ops, orc, synth):
    """lens[b] == 0 is an empty sequence, as for the attention call: its q row comes back zero and
    nothing is written to its part of the cache; the other rows are unaffected."""
    cfg = synth.tiny_config(2048)
    D, n_q, n_kv, cap, B = cfg.head_dim, cfg.n_attn_heads, cfg.n_kv_heads, 64, 3
    rng = np.random.default_rng(9)
    qkv = torch.from_numpy(rng.standard_normal((B, (n_q + 2 * n_kv) * D)).astype(np.float32)).cuda()
    cs, sn = orc.rope_tables(cfg, 8)
    cs_d, sn_d = torch.from_numpy(cs).cuda(), torch.from_numpy(sn).cuda()
    both = []
    for lens in ([3, 0, 5], [3, 2, 5]):
        cache = ops.KVCache(B, n_kv, D, cap)
        cache.kv.view(torch.int16).fill_(0x1234)
        q = ops.rope_kv_store(qkv, cache, cs_d, sn_d, torch.tensor(lens, dtype=torch.int32).cuda(), n_q)
        torch.cuda.synchronize()
        both.append((q.cpu().numpy(), cache.kv.view(torch.int16).cpu().numpy().reshape(B, -1)))
    (q0, kv0), (q1, kv1) = both
    assert (q0[1] == 0).all() and (kv0[1] == 0x1234).all()           # empty row: zero q, cache untouched
    assert (kv1[1] != 0x1234).any()                                   # the same row with a length does store
    for b in (0, 2):
        assert np.array_equal(q0[b], q1[b]) and np.array_equal(kv0[b], kv1[b])


@pytest.mark.parametrize("D,n_q,n_kv", [(32, 4, 4), (32, 8, 2), (64, 64, 8), (64, 6, 3)])
def test_rotation_of_few_rows_equals_that_of_many(ops, D, n_q, n_kv):
    """Few rows have several workgroups each; at 300 a row has one."""
    g = torch.Generator(device="cuda").manual_seed(D + n_q)
    B, n = 300, 70
    qkv = torch.randn(B, (n_q + 2 * n_kv) * D, generator=g, device="cuda")
    cs, sn = (torch.randn(n, D // 2, generator=g, device="cuda") for _ in range(2))
    lens = torch.randint(0, n + 1, (B,), generator=g, device="cuda", dtype=torch.int32)

    def rotate(rows):
        cache = ops.KVCache(rows, n_kv, D, 128)
        cache.kv.view(torch.int16).fill_(0x1234)
        return ops.rope_kv_store(qkv[:rows].contiguous(), cache, cs, sn, lens[:rows].contiguous(), n_q), cache.kv.view(torch.int16).view(rows, -1)

    q, kv = rotate(B)
    for rows in (1, 2, 25, 26, 42, 43, 64, 65, 128, 129):
        q_few, kv_few = rotate(rows)
        assert torch.equal(q_few.view(rows, -1), q[:rows].view(rows, -1)) and torch.equal(kv_few, kv[:rows]), rows


def _internal(name, argtypes):
    """A function of namespace gptoss without a C entry point, by its linker name."""
    import ctypes as C
    from conftest import load_pkg
    lib = load_pkg("lib")
    f = getattr(lib.load(), name)
    f.restype, f.argtypes = C.c_int, argtypes
    return lambda *a: lib.check(f(*a, torch.cuda.current_stream().cuda_stream))


# H: one 16-byte piece, part of a wave, one wave short of / just past a piece of 256 threads, an odd number of pieces, the last
# instance; sums: one, a group of four behind it and one more, ...
@pytest.mark.parametrize("H", [4, 64, 252, 1020, 1024, 1028, 2044, 2052, 2880, 4096, 4100, 8192, 8196, 16384])
@pytest.mark.parametrize("parts,layer", [(1, 0), (2, 2), (5, 3), (6, 4), (16, 8)])
def test_depth_average_and_norm(ops, H, parts, layer):
    import ctypes as C
    P, I = C.c_void_p, C.c_int
    run = _internal("_ZN6gptoss22run_depth_average_normEPfPKfiS0_mS2_iS2_PtS0_iifiP12ihipStream_t",
                    [P, P, I, P, C.c_size_t, P, I, P, P, P, I, I, C.c_float, I, P])
    g = torch.Generator(device="cuda").manual_seed(H + parts)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    rows, plane = 3, 5 * H
    x, y, w = rnd(rows, H), rnd(parts, rows, H), rnd(H)
    history, weights = rnd(layer + 3, 5, H), rnd(layer + 2)
    before, own = history.clone(), x.double() + y.double().sum(0)
    size = x.double().abs() + y.double().abs().sum(0)
    t16, t32 = torch.empty(rows, H, device="cuda", dtype=torch.bfloat16), torch.empty(rows, H, device="cuda")
    run(x.data_ptr(), y.data_ptr(), parts, history.data_ptr(), plane, weights.data_ptr(), layer, w.data_ptr(), t16.data_ptr(),
        t32.data_ptr(), rows, H, 1e-5, H)
    # a sum of n fp32 terms: each of up to n roundings is at most 2^-24 of the sum of their sizes
    assert bool(((history[layer + 1, :rows].double() - own).abs() <= size * (parts + 1) * 2.0 ** -24).all())
    terms = weights[:layer + 1, None, None].double() * before[:layer + 1, :rows].double()
    want = terms.sum(0) + weights[layer + 1].double() * own
    bound = (terms.abs().sum(0) + weights[layer + 1].double().abs() * size) * (layer + parts + 4) * 2.0 ** -24
    assert bool(((x.double() - want).abs() <= bound).all())
    scale = w.double() / torch.sqrt((x.double() ** 2).mean(-1, keepdim=True) + 1e-5)
    # squares, their root and its reciprocal in fp32, one more rounding: 2^-21 of the result; bf16: 2^-8
    assert bool(((t32.double() - x.double() * scale).abs() <= (x.double() * scale).abs() * 2.0 ** -21 + 1e-30).all())
    assert torch.equal(t16, t32.bfloat16())
    history[layer + 1, :rows] = before[layer + 1, :rows]
    assert torch.equal(history, before)      # nothing else is written


# bf16 rows from 1024 elements on and fp32 rows from 512 on go 16 bytes at a time, if whole and aligned
@pytest.mark.parametrize("dtype,H,ld", [("bf16", 1016, 1016), ("bf16", 1024, 1024), ("bf16", 1020, 1024), ("bf16", 1024, 1028), ("bf16", 2048, 2112),
                                        ("bf16", 64, 1024), ("f32", 508, 508), ("f32", 512, 512), ("f32", 510, 512), ("f32", 1028, 1088)])
@pytest.mark.parametrize("with_positions", [False, True])
def test_embedding_rows(ops, dtype, H, ld, with_positions):
    import ctypes as C
    name = {"bf16": "_ZN6gptoss22run_embedding_positionEPKtS1_PKiS3_PfS4_iiiiiP12ihipStream_t",
            "f32": "_ZN6gptoss26run_embedding_position_f32EPKfS1_PKiS3_PfS4_iiiiiP12ihipStream_t"}[dtype]
    run = _internal(name, [C.c_void_p] * 6 + [C.c_int] * 5 + [C.c_void_p])
    g = torch.Generator(device="cuda").manual_seed(H)
    cast = (lambda v: v.bfloat16()) if dtype == "bf16" else (lambda v: v)
    V, n_pos, rows = 37, 11, 5
    flat = cast(torch.randn(V * H + 1, generator=g, device="cuda"))
    positions = cast(torch.randn(n_pos, H, generator=g, device="cuda"))
    tokens = torch.tensor([0, V - 1, 5, V + 3, -1], dtype=torch.int32, device="cuda")   # outside: clamped
    lens = torch.tensor([1, n_pos, n_pos + 4, 3, 0], dtype=torch.int32, device="cuda")
    for shift in (0, 1):   # a table that no wide load may touch
        table = flat[shift:shift + V * H].view(V, H)
        x = torch.full((rows, ld), 7.0, device="cuda")
        x0 = torch.full_like(x, 7.0)
        run(table.data_ptr(), positions.data_ptr() if with_positions else None, tokens.data_ptr(), lens.data_ptr(), x.data_ptr(),
            x0.data_ptr() if with_positions else None, rows, H, ld, V, n_pos)
        want = torch.zeros(rows, ld, device="cuda")
        want[:, :H] = table[tokens.long().clamp(0, V - 1)].float()
        if with_positions:
            want[:, :H] += positions[(lens.long() - 1).clamp(0, n_pos - 1)].float()
            assert torch.equal(x0, want)
        assert torch.equal(x, want), shift


# lengths at the edges of 16-slot rows, blocks, chunks; one and two chunks; a ring that has wrapped; an empty sequence
@pytest.mark.parametrize("D,n_q,n_kv,cap,window,lens", [
    (64, 64, 8, 576, 0, (1, 16, 17, 63, 64)), (64, 16, 2, 1088, 0, (65, 512, 513, 0, 577, 1088)), (64, 4, 4, 192, 128, (128, 129, 190)),
    (64, 16, 1, 128, 128, (127, 128, 129, 300, 384)), (32, 24, 3, 640, 0, (5, 33, 600)), (32, 8, 8, 64, 64, (64, 65, 200)),
])
def test_rotation_within_the_attention_equals_that_in_front_of_it(ops, D, n_q, n_kv, cap, window, lens):
    """gptoss::attn_decode_rope by its linker name: one kernel where no two rows are of one sequence, two otherwise."""
    import ctypes as C
    from conftest import load_pkg
    f = load_pkg("lib").load()._ZN6gptoss16attn_decode_ropeEPKfPfS1_S1_PvPKiS1_S3_ibiiiiiiS3_mS3_S5_
    p, i = C.c_void_p, C.c_int
    f.argtypes = [p, p, p, p, p, p, p, p, i, C.c_bool, i, i, i, i, i, i, p, C.c_size_t, p, p]
    g = torch.Generator(device="cuda").manual_seed(D + cap)
    B, slots = len(lens), len(lens) + 2
    qkv = torch.randn(B, (n_q + 2 * n_kv) * D, device="cuda", generator=g)
    angle = torch.rand(1200, D // 2, device="cuda", generator=g) * 6.3
    cos, sin, sinks = angle.cos(), angle.sin(), torch.randn(n_q, device="cuda", generator=g)
    filled = torch.randn(slots * n_kv * cap * 2 * D, device="cuda", generator=g).to(torch.bfloat16)
    lens_t = torch.tensor(lens, dtype=torch.int32, device="cuda")
    seq_map = torch.randperm(slots, device="cuda", generator=g)[:B].to(torch.int32)
    ws = torch.empty(1 << 24, dtype=torch.uint8, device="cuda")
    got = []
    for own in (False, True):
        kv, out = filled.clone(), torch.zeros(B, n_q, D, dtype=torch.bfloat16, device="cuda")
        q = torch.full((B, n_q, D), 7.0, device="cuda")
        torch.cuda.synchronize()
        assert f(qkv.data_ptr(), q.data_ptr(), cos.data_ptr(), sin.data_ptr(), kv.data_ptr(), lens_t.data_ptr(), sinks.data_ptr(),
                 out.data_ptr(), B, own, n_q, n_kv, D, cap, window, max(lens), ws.data_ptr(), ws.numel(), None,
                 seq_map.data_ptr()) == 0
        torch.cuda.synchronize()
        assert bool((q == 7.0).all()) == own            # the queries in front of it go through memory
        got.append((out, kv))
    assert torch.equal(got[0][0].view(torch.int16), got[1][0].view(torch.int16))
    assert torch.equal(got[0][1].view(torch.int16), got[1][1].view(torch.int16)) and not torch.equal(filled, got[1][1])


def test_calls_go_to_the_current_stream(ops, monkeypatch):
    def streams():
        torch.cuda.init()
        other = torch.cuda.Stream()
        with torch.cuda.stream(other):
            inside = ops._stream(), other.cuda_stream
        return [inside, (ops._stream(), torch.cuda.current_stream().cuda_stream)]
    for have, want in streams():
        assert have == want
    monkeypatch.setattr(ops, "_raw_stream", None)      # a torch without it
    for have, want in streams():
        assert have == want
