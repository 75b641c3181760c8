"""GPU parity of decode attention (sinks, sliding window, GQA, ragged lengths, ring cache)
against the CPU oracle, through the C ABI."""
import math

import numpy as np
import pytest
import torch

from conftest import TOL_MAX, TOL_MEAN, rel_errors

pytestmark = pytest.mark.gpu


def _mk(B, S, n_q, n_kv, D, seed):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(B, n_q, D, generator=g)
    K = torch.randn(B, S, n_kv, D, generator=g).to(torch.bfloat16)
    V = torch.randn(B, S, n_kv, D, generator=g).to(torch.bfloat16)
    sinks = torch.randn(n_q, generator=g)
    return q, K, V, sinks


def _run(ops, q, K, V, lens, sinks, window, capacity=None, max_len=None):
    B, S, n_kv, D = K.shape
    n_q = q.shape[1]
    cap = capacity or ((S + 63) // 64 * 64)
    cache = ops.KVCache(B, n_kv, D, cap)
    # never-written slots keep whatever the allocator left there, NaN patterns included
    cache.kv.view(torch.int16).fill_(0x7FC1)
    cache.write(K.cuda(), V.cuda(), 0)
    attn = ops.AttnDecode(B, n_q, n_kv, D, max_len or int(lens.max()))
    out = attn.forward(q.cuda(), cache, torch.as_tensor(lens, dtype=torch.int32).cuda(),
                       None if sinks is None else sinks.cuda(), window=window)
    torch.cuda.synchronize()
    return out.float().cpu().numpy()


@pytest.mark.parametrize("B,n_q,n_kv,D,lens,window", [
    (3, 8, 2, 32, [1, 2, 63], 0),                    # tiny-model heads, very short contexts
    (4, 8, 2, 32, [64, 65, 127, 128], 0),
    (4, 8, 2, 32, [100, 129, 200, 300], 128),        # window smaller than the context
    (5, 64, 8, 64, [1, 17, 256, 257, 700], 0),       # 20B heads, one and several chunks
    (3, 64, 8, 64, [512, 1500, 4096], 0),            # long contexts: 512-token chunks + merge
    (4, 64, 8, 64, [100, 128, 129, 4000], 128),      # sliding window on a full-length cache
    (2, 16, 1, 64, [333, 90], 0),                    # 16 query heads per kv head
    (2, 4, 4, 64, [70, 5], 0),                       # no sharing (MHA)
])
def test_attn_matches_oracle(ops, orc, B, n_q, n_kv, D, lens, window):
    lens = np.asarray(lens, np.int32)
    S = int(lens.max())
    q, K, V, sinks = _mk(B, S, n_q, n_kv, D, seed=S + n_q)
    got = _run(ops, q, K, V, lens, sinks, window)
    want = orc.attn_decode(q.numpy(), K.float().numpy(), V.float().numpy(), lens, sinks.numpy(), window)
    assert np.isfinite(got).all()
    mx, mean = rel_errors(got, want)
    assert mx <= TOL_MAX and mean <= TOL_MEAN, (mx, mean)


def test_attn_no_sink_equals_sdpa(ops):
    """sinks=None reduces to plain softmax attention (checked against torch SDPA)."""
    B, n_q, n_kv, D, S = 2, 64, 8, 64, 300
    q, K, V, _ = _mk(B, S, n_q, n_kv, D, seed=11)
    lens = np.array([S, S], np.int32)
    got = _run(ops, q, K, V, lens, None, 0)
    Kf = K.float().permute(0, 2, 1, 3).repeat_interleave(n_q // n_kv, dim=1)
    Vf = V.float().permute(0, 2, 1, 3).repeat_interleave(n_q // n_kv, dim=1)
    want = torch.nn.functional.scaled_dot_product_attention(q.unsqueeze(2), Kf, Vf).squeeze(2).numpy()
    mx, mean = rel_errors(got, want)
    assert mx <= TOL_MAX and mean <= TOL_MEAN, (mx, mean)


def test_attn_ring_cache_wrapped(ops, orc):
    """A cache of capacity == window holds position p in slot p % capacity; after wrapping the
    result equals attention over the last `window` positions."""
    B, n_q, n_kv, D, W = 3, 8, 2, 32, 128
    total = [130, 256, 301]
    S = max(total)
    q, K, V, sinks = _mk(B, S, n_q, n_kv, D, seed=5)
    cache = ops.KVCache(B, n_kv, D, W)
    Kc, Vc = K.cuda(), V.cuda()
    for p0 in range(0, S, 64):                          # stream the positions through the ring
        n = min(64, S - p0)
        cache.write(Kc[:, p0:p0 + n], Vc[:, p0:p0 + n], p0)
    torch.cuda.synchronize()
    # sequences shorter than S saw extra writes; rebuild per-sequence caches for exactness
    outs = []
    for b in range(B):
        cb = ops.KVCache(1, n_kv, D, W)
        for p0 in range(0, total[b], 50):
            n = min(50, total[b] - p0)
            cb.write(Kc[b:b + 1, p0:p0 + n], Vc[b:b + 1, p0:p0 + n], p0)
        attn = ops.AttnDecode(1, n_q, n_kv, D, max_len=2048)
        o = attn.forward(q[b:b + 1].cuda(), cb, torch.tensor([total[b]], dtype=torch.int32).cuda(),
                         sinks.cuda(), window=W)
        outs.append(o.float().cpu().numpy())
    got = np.concatenate(outs)
    want = orc.attn_decode(q.numpy(), K.float().numpy(), V.float().numpy(),
                           np.asarray(total, np.int32), sinks.numpy(), W)
    mx, mean = rel_errors(got, want)
    assert mx <= TOL_MAX and mean <= TOL_MEAN, (mx, mean)


def test_attn_len1_closed_form(ops):
    """One cached position: o = v * e^s / (e^s + e^sink)."""
    B, n_q, n_kv, D = 2, 8, 2, 32
    q, K, V, sinks = _mk(B, 1, n_q, n_kv, D, seed=3)
    got = _run(ops, q, K, V, np.array([1, 1], np.int32), sinks, 0)
    Kf, Vf = K.float().numpy(), V.float().numpy()
    for b in range(B):
        for h in range(n_q):
            g = h // (n_q // n_kv)
            s = float(q[b, h].numpy() @ Kf[b, 0, g]) / np.sqrt(D)
            w = np.exp(s) / (np.exp(s) + np.exp(float(sinks[h])))
            np.testing.assert_allclose(got[b, h], w * Vf[b, 0, g], rtol=1e-2, atol=1e-2)


def test_attn_without_lengths_means_every_row_has_max_len(ops):
    """lens = NULL (lock-step decoding: the host knows the one length) gives the bits of an array filled
    with max_len, in both launch forms."""
    for B, n_q, n_kv, D, S, L in ((5, 8, 2, 32, 256, 200), (70, 64, 8, 64, 640, 601)):
        q, K, V, sinks = _mk(B, S, n_q, n_kv, D, seed=21)
        cache = ops.KVCache(B, n_kv, D, S)
        cache.write(K.cuda(), V.cuda(), 0)
        attn = ops.AttnDecode(B, n_q, n_kv, D, S)
        lens = torch.full((B,), L, dtype=torch.int32, device="cuda")
        for window in (0, 128):
            a = attn.forward(q.cuda(), cache, lens, sinks.cuda(), window=window, max_len=L).clone()
            b = attn.forward(q.cuda(), cache, None, sinks.cuda(), window=window, max_len=L)
            assert torch.equal(a, b), (B, window)


def test_attn_output_rows_kept_back_equal_rows_stored_at_once(ops):
    """One query row per sequence and contexts of one chunk run on a resident grid that keeps its
    output rows in LDS and writes them 16 bytes at a time after its last row; an output buffer that
    is only 8-byte aligned gets the plain launch, which stores every row as it is finished.  Same bits
    for a few rows (less than one round of the grid), for 1200 and for 8000 workgroup indices (several
    rounds; the last case fills a workgroup's 16 slots and makes it write them in between), with
    ragged lengths, empty rows and both head sizes."""
    for B, n_q, n_kv, D, S in ((3, 8, 2, 32, 128), (600, 16, 8, 64, 192), (4000, 8, 8, 32, 128)):
        q, K, V, sinks = _mk(B, S, n_q, n_kv, D, seed=33)
        cache = ops.KVCache(B, n_kv, D, S)
        cache.write(K.cuda(), V.cuda(), 0)
        attn = ops.AttnDecode(B, n_q, n_kv, D, S)
        g = torch.Generator().manual_seed(7)
        lens = torch.randint(0, S + 1, (B,), generator=g, dtype=torch.int32)
        lens[0] = S
        lens = lens.cuda()
        flat = torch.zeros(B * n_q * D + 8, dtype=torch.bfloat16, device="cuda")
        for window in (0, 64):
            a = attn.forward(q.cuda(), cache, lens, sinks.cuda(), window=window)
            off = flat[4:4 + B * n_q * D].view(B, n_q, D)   # 8 bytes past a 16-byte boundary
            assert off.data_ptr() % 16 == 8
            attn.forward(q.cuda(), cache, lens, sinks.cuda(), window=window, out=off)
            assert torch.equal(a, off), (B, D, window)


def test_attn_bad_arguments(ops):
    import ctypes as C
    from conftest import load_pkg
    lib = load_pkg("lib")
    L = lib.load(strict=False)
    q = torch.zeros(1, 8, 48, device="cuda")
    rc = L.gptoss_attn_decode(C.c_void_p(q.data_ptr()), C.c_void_p(q.data_ptr()), C.c_void_p(q.data_ptr()),
                              None, C.c_void_p(q.data_ptr()), 1, 8, 2, 48, 64, 0,
                              10, C.c_void_p(q.data_ptr()), 1 << 20, None)
    assert rc == 2 and "head_dim" in lib.last_error()
    rc = L.gptoss_attn_decode(None, None, None, None, None, 1, 8, 2, 64, 64, 0, 10, None, 0, None)
    assert rc == 1


def test_attn_many_long_sequences_static_and_ticket_rounds(ops, orc):
    """160 sequences x 8 kv heads: enough for the workgroup-per-row kernel (long rows: four waves
    interleave 64-slot blocks, longest rows first) next to the one-wave kernel (rows of up to 512
    slots); lengths from 0 to the full 4096, the result twice in a row from the same workspace."""
    B, n_q, n_kv, D, S = 160, 16, 8, 64, 4096
    rng = np.random.default_rng(42)
    lens = rng.integers(1, S + 1, size=B).astype(np.int32)
    lens[:4] = [0, 1, S, 513]
    q, K, V, sinks = _mk(B, S, n_q, n_kv, D, seed=3)
    cache = ops.KVCache(B, n_kv, D, S)
    cache.kv.view(torch.int16).fill_(0x7FC1)
    cache.write(K.cuda(), V.cuda(), 0)
    attn = ops.AttnDecode(B, n_q, n_kv, D, S)
    lens_d = torch.as_tensor(lens).cuda()
    a = attn.forward(q.cuda(), cache, lens_d, sinks.cuda(), window=0).float().cpu().numpy()
    b = attn.forward(q.cuda(), cache, lens_d, sinks.cuda(), window=0).float().cpu().numpy()
    assert np.array_equal(a, b)                       # whatever order the rows were dealt in
    want = orc.attn_decode(q.numpy(), K.float().numpy(), V.float().numpy(), lens, sinks.numpy(), 0)
    assert np.isfinite(a).all()
    mx, mean = rel_errors(a, want)
    assert mx <= TOL_MAX and mean <= TOL_MEAN, (mx, mean)
    # the same rows through the other launch form: 32 sequences x 8 kv heads is below the switch, so
    # long rows are 512-slot chunks merged by the reduce kernel.  Rows of one chunk take the same
    # path in both calls (equal bits); longer rows are summed in another order and may differ by a
    # last-bit rounding of the bf16 output here and there.
    n = 32
    few = ops.AttnDecode(n, n_q, n_kv, D, S)
    c = few.forward(q[:n].cuda().contiguous(), cache.first(n), lens_d[:n].contiguous(), sinks.cuda(),
                    window=0).float().cpu().numpy()
    short = lens[:n] <= 512
    assert short.any() and (~short).any()
    assert np.array_equal(a[:n][short], c[short])
    diff = np.abs(a[:n] - c)
    assert diff.max() <= 2.0 ** -7 * np.abs(c).max(), diff.max()
    assert (diff > 0).mean() < 0.02, (diff > 0).mean()


def test_attn_batch_larger_than_one_launch_slice(ops, orc):
    """More sequences than one launch keeps in LDS (2048): the call is sliced internally."""
    B, n_q, n_kv, D, S = 2100, 2, 1, 32, 64
    rng = np.random.default_rng(7)
    lens = rng.integers(1, S + 1, size=B).astype(np.int32)
    q, K, V, sinks = _mk(B, S, n_q, n_kv, D, seed=9)
    got = _run(ops, q, K, V, lens, sinks, 0)
    want = orc.attn_decode(q.numpy(), K.float().numpy(), V.float().numpy(), lens, sinks.numpy(), 0)
    mx, mean = rel_errors(got, want)
    assert mx <= TOL_MAX and mean <= TOL_MEAN, (mx, mean)


@pytest.mark.parametrize("B,T,pos0,n_q,n_kv,D,window", [
    (3, 40, 0, 8, 2, 32, 0),          # tiny-model heads, whole prompt from position 0
    (2, 128, 0, 64, 8, 64, 128),      # 20B heads, the window exactly as long as the prompt
    (2, 300, 0, 64, 8, 64, 128),      # prompt longer than the window (linear cache)
    (2, 70, 500, 64, 8, 64, 0),       # a later slice of a long context: two chunks per row
    (1, 200, 1000, 64, 8, 64, 0),     # rows on both sides of the 1024-position chunk-size change
    (2, 65, 60, 64, 8, 64, 128),      # odd row count (the last row of a sequence has no partner), window edges
    (3, 41, 0, 8, 2, 32, 0),          # odd row count, four query heads per kv head
    (1, 66, 480, 64, 8, 64, 0),       # partners on either side of a chunk boundary (512 / 513 positions)
    (1, 1024, 0, 64, 8, 64, 0),       # the reference's longest prompt: 16 blocks per row group
    (2, 1024, 0, 8, 2, 32, 128),      # the same with the window, head_dim 32
    (1, 1000, 24, 16, 2, 64, 128),    # row groups that start inside a block, 8 query heads per kv head, ragged end
    (2, 20, 0, 8, 2, 32, 0),          # fewer than 32 positions: the row-pair form
])
def test_attn_prefill_rows_equal_decode_calls(ops, orc, B, T, pos0, n_q, n_kv, D, window):
    """Prompt attention = the decode attention of every position at once: row (b, t) must equal, bit
    for bit, the decode call with lens = pos0 + t + 1 on the same cache (whatever else is in the
    launch) while the row's slot range fits one 512-slot chunk; a longer row is summed block by
    block in one pass where the decode call merges chunk partials, so it may differ from it by a
    last-bit rounding of a few outputs.  A sample of rows must match the oracle."""
    S = pos0 + T
    g = torch.Generator().manual_seed(S + n_q)
    q = torch.randn(B, T, n_q, D, generator=g)
    K = torch.randn(B, S, n_kv, D, generator=g).to(torch.bfloat16)
    V = torch.randn(B, S, n_kv, D, generator=g).to(torch.bfloat16)
    sinks = torch.randn(n_q, generator=g)
    cap = (S + 63) // 64 * 64
    cache = ops.KVCache(B, n_kv, D, cap)
    cache.kv.view(torch.int16).fill_(0x7FC1)
    cache.write(K.cuda(), V.cuda(), 0)
    pre = ops.AttnPrefill(B, T, n_q, n_kv, D, S)
    got = pre.forward(q.cuda(), cache, pos0=pos0, sinks=sinks.cuda(), window=window)
    torch.cuda.synchronize()
    assert torch.isfinite(got.float()).all()
    dec = ops.AttnDecode(B, n_q, n_kv, D, S)
    # every row of the short prompts (two consecutive rows share a wave), a sample of the long ones
    for t in (range(T) if T <= 70 else sorted({0, 1, T // 3, T // 2, T - 2, T - 1})):
        lens = torch.full((B,), pos0 + t + 1, dtype=torch.int32)
        one = dec.forward(q[:, t].contiguous().cuda(), cache, lens.cuda(), sinks.cuda(), window=window,
                          max_len=pos0 + t + 1)
        length = pos0 + t + 1
        first_slot = (max(0, length - window) if window else 0) // 64 * 64
        if length - first_slot <= 512:
            assert torch.equal(got[:, t], one), t
        else:
            a, b = got[:, t].float(), one.float()
            assert (a - b).abs().max() <= 2.0 ** -7 * b.abs().max(), t        # one bf16 step at the largest output
            assert (a != b).float().mean() < 0.05, t
        want = orc.attn_decode(q[:, t].numpy(), K.float().numpy(), V.float().numpy(), lens.numpy(), sinks.numpy(),
                               window)
        mx, mean = rel_errors(got[:, t].float().cpu().numpy(), want)
        assert mx <= TOL_MAX and mean <= TOL_MEAN, (t, mx, mean)


def test_attn_prefill_refuses_a_wrapped_window_ring(ops):
    from conftest import load_pkg
    lib = load_pkg("lib")
    cache = ops.KVCache(1, 8, 64, 128)
    pre = ops.AttnPrefill(1, 200, 64, 8, 64, 200)
    with pytest.raises(lib.GptossError):
        pre.forward(torch.zeros(1, 200, 64, 64).cuda(), cache, window=128)


@pytest.mark.parametrize("n_q,n_kv,D,cap,window", [
    (64, 8, 64, 512, 0), (64, 8, 64, 512, 128), (64, 8, 64, 128, 128),   # 20B heads; window; a ring that has wrapped
    (64, 8, 64, 192, 128),                                               # a wrapped ring longer than its window
    (8, 8, 64, 512, 0), (32, 8, 32, 512, 0), (96, 8, 64, 512, 200),      # 1, 4 and 12 query heads per kv head
])
def test_a_few_rows_have_the_bits_of_the_same_rows_among_many(ops, n_q, n_kv, D, cap, window):
    """Rows of up to 512 slots: a workgroup each where few are served, a wave each where many are."""
    B = 160                                              # 1280 (row, kv head) pairs
    g = torch.Generator(device="cuda").manual_seed(n_q + cap + window)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)
    longest = cap if not (window and cap < 512) else cap + 100
    edges = [0, 1, 2, 63, 64, 65, 127, 128, 129, 255, 257, 448, 449, 511, 512]
    lens = [min(x, longest) for x in edges] + torch.randint(1, longest + 1, (B - len(edges),), generator=g, device="cuda").tolist()
    lens = torch.tensor(lens, dtype=torch.int32, device="cuda")
    cache = ops.KVCache(B, n_kv, D, cap)
    cache.kv.view(torch.int16).fill_(0x7FC1)             # NaN patterns where nothing is written
    filled = min(int(lens.max()), cap)
    cache.write(rnd(B, filled, n_kv, D).bfloat16(), rnd(B, filled, n_kv, D).bfloat16(), 0)
    q, sinks = rnd(B, n_q, D) * 2, rnd(n_q)
    many = ops.AttnDecode(B, n_q, n_kv, D, longest).forward(q, cache, lens, sinks, window=window)
    for rows in (1, 7, 15, 100):
        few = ops.AttnDecode(rows, n_q, n_kv, D, longest).forward(q[:rows].contiguous(), cache.first(rows), lens[:rows], sinks,
                                                                  window=window)
        assert torch.equal(few.view(torch.int16), many[:rows].view(torch.int16)), rows


def _kernels(ops, call):
    with ops.KernelTrace(capacity=16) as trace:
        call()
    return [name for name, _ in trace.results()]


# longest: rows of one chunk or of up to five; a window over them; a ring that has wrapped
@pytest.mark.parametrize("longest,cap,window", [(2000, 2048, 0), (700, 768, 0), (2000, 2048, 700), (3000, 1024, 600)])
@pytest.mark.parametrize("n_q,n_kv,D", [(64, 8, 64), (96, 8, 64), (64, 8, 32)])
def test_few_rows_of_several_chunks_have_the_bits_of_the_same_rows_among_more(ops, n_q, n_kv, D, longest, cap, window):
    """All loads of a chunk at once where few are served; for 60 rows heads of 64 three workgroups per CU, heads of 32 a wave per
    chunk."""
    B = 60
    g = torch.Generator(device="cuda").manual_seed(longest + window)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)
    edges = [longest, 513, 512, 511, 1024, 1025, 64, 1, 0]
    lens = [min(x, longest) for x in edges] + torch.randint(1, longest + 1, (B - len(edges),), generator=g, device="cuda").tolist()
    lens = torch.tensor(lens, dtype=torch.int32, device="cuda")
    cache = ops.KVCache(B, n_kv, D, cap)
    cache.write(rnd(B, cap, n_kv, D).bfloat16(), rnd(B, cap, n_kv, D).bfloat16(), 0)
    q, sinks = rnd(B, n_q, D) * 2, rnd(n_q)
    out = {}
    def attend(rows):
        attn = ops.AttnDecode(rows, n_q, n_kv, D, longest)
        out[rows] = attn.forward(q[:rows].contiguous(), cache.first(rows), lens[:rows], sinks, window=window)
    assert _kernels(ops, lambda: attend(B)) == ["attn_decode", "attn_reduce"]
    for rows in (1, 2, 5, 9):
        assert _kernels(ops, lambda: attend(rows)) == ["attn_decode_few", "attn_reduce"], rows
        assert torch.equal(out[rows].view(torch.int16), out[B][:rows].view(torch.int16)), rows


# rounds of 1024 (row, kv head, chunk) items that are nearly full, and one that is not (24 of 2000: 768)
@pytest.mark.parametrize("B,longest", [(32, 2000), (63, 1000), (63, 2000), (48, 3900), (24, 2000)])
def test_rows_of_one_length_have_the_same_bits_a_workgroup_or_a_wave_per_chunk(ops, B, longest):
    """Without lengths all rows are known to have the longest one, and go by a wave per chunk where that fills rounds."""
    n_q, n_kv, D, cap = 64, 8, 64, (longest + 63) // 64 * 64
    g = torch.Generator(device="cuda").manual_seed(longest + B)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)
    cache = ops.KVCache(B, n_kv, D, cap)
    cache.kv.view(torch.int16).fill_(0x7FC1)             # NaN patterns where nothing is written
    cache.write(rnd(B, longest, n_kv, D).bfloat16(), rnd(B, longest, n_kv, D).bfloat16(), 0)
    q, sinks = rnd(B, n_q, D) * 2, rnd(n_q)
    attn = ops.AttnDecode(B, n_q, n_kv, D, longest)
    known = attn.forward(q, cache, None, sinks)
    given = attn.forward(q, cache, torch.full((B,), longest, dtype=torch.int32, device="cuda"), sinks)
    assert torch.isfinite(known).all() and torch.equal(known.view(torch.int16), given.view(torch.int16))


# rows of one chunk: up to 512 sequences a workgroup each, 520 a wave, short ones up to 80 and 90; of one chunk and of several: up to
# 1024 sequences a workgroup for each of one chunk as well, in front of the kernel that takes the others, 1030 a wave
@pytest.mark.parametrize("sequences,longest,cap,window", [
    ((90, 33, 64, 65, 80), 128, 128, 0), ((90, 64, 80), 400, 512, 100), ((520, 65, 200, 512), 192, 192, 0),
    ((520, 65, 200, 512), 512, 512, 0), ((520, 65, 512), 512, 512, 300),
    ((1030, 64, 65, 300, 1024), 700, 704, 0), ((1030, 64, 1024), 900, 640, 576)])
def test_rows_have_the_same_bits_a_workgroup_or_a_wave_each(ops, sequences, longest, cap, window):
    B, n_q, n_kv, D = sequences[0], 64, 8, 64
    g = torch.Generator(device="cuda").manual_seed(longest + window)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)
    edges = [longest, 0, 1, 64, 65, 255, 256, 257, 448, 449, 511, 512, 513]
    lens = [min(x, longest) for x in edges] + torch.randint(1, longest + 1, (B - len(edges),), generator=g, device="cuda").tolist()
    lens = torch.tensor(lens, dtype=torch.int32, device="cuda")
    cache = ops.KVCache(B, n_kv, D, cap)
    cache.kv.view(torch.int16).fill_(0x7FC1)             # NaN patterns where nothing is written
    cache.write(rnd(B, min(longest, cap), n_kv, D).bfloat16(), rnd(B, min(longest, cap), n_kv, D).bfloat16(), 0)
    q, sinks = rnd(B, n_q, D) * 2, rnd(n_q)
    out = {}
    for rows in sequences:
        attn = ops.AttnDecode(rows, n_q, n_kv, D, longest)
        out[rows] = attn.forward(q[:rows].contiguous(), cache.first(rows), lens[:rows], sinks, window=window)
        assert torch.isfinite(out[rows]).all()
        assert torch.equal(out[rows].view(torch.int16), out[B][:rows].view(torch.int16)), rows


@pytest.mark.parametrize("pos0,T", [(0, 130), (500, 70), (900, 9)])
def test_prompt_rows_of_more_than_eight_heads_per_kv_head(ops, pos0, T):
    """They go row by row: thousands of rows are many, however few the sequences are."""
    n_q, n_kv, D = 96, 8, 64
    n = pos0 + T
    g = torch.Generator(device="cuda").manual_seed(T)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)
    k, v, q, sinks = rnd(1, n, n_kv, D).bfloat16(), rnd(1, n, n_kv, D).bfloat16(), rnd(1, T, n_q, D), rnd(n_q)
    cache = ops.KVCache(1, n_kv, D, (n + 63) // 64 * 64)
    cache.write(k, v)
    prefill, out = ops.AttnPrefill(1, T, n_q, n_kv, D, n), []
    names = _kernels(ops, lambda: out.append(prefill.forward(q, cache, pos0=pos0, sinks=sinks)))
    # up to 512 items: T rows of 8 kv heads and one or two chunks
    assert names[0] == ("attn_decode_few" if T * 8 * -(-n // 512) <= 512 else "attn_decode"), names
    one = ops.AttnDecode(1, n_q, n_kv, D, n)
    for t in (0, 1, T // 2, T - 1):
        lens = torch.tensor([pos0 + t + 1], dtype=torch.int32, device="cuda")
        want = one.forward(q[:, t].contiguous(), cache, lens, sinks)
        assert torch.equal(out[0][:, t].view(torch.int16), want.view(torch.int16)), t


@pytest.mark.parametrize("B", [70, 250])       # 560 and 2000 (row, kv head) pairs: less than a round of the resident grid's waves
def test_attn_output_rows_kept_back_in_less_than_one_round(ops, B):
    """As above, where every wave has one row at most and the rows are still too many for a workgroup each."""
    n_q, n_kv, D, S = 16, 8, 64, 192
    q, K, V, sinks = _mk(B, S, n_q, n_kv, D, seed=34)
    cache = ops.KVCache(B, n_kv, D, S)
    cache.write(K.cuda(), V.cuda(), 0)
    attn = ops.AttnDecode(B, n_q, n_kv, D, S)
    lens = torch.randint(0, S + 1, (B,), generator=torch.Generator().manual_seed(7), dtype=torch.int32).cuda()
    flat, out = torch.zeros(B * n_q * D + 8, dtype=torch.bfloat16, device="cuda"), []
    assert _kernels(ops, lambda: out.append(attn.forward(q.cuda(), cache, lens, sinks.cuda()))) == ["attn_decode"]
    off = flat[4:4 + B * n_q * D].view(B, n_q, D)
    attn.forward(q.cuda(), cache, lens, sinks.cuda(), out=off)
    assert torch.equal(out[0], off)


# (sequences, positions, new positions per sequence or 0 for decoding): a workgroup per chunk without and with a merge, a
# wave per row, a workgroup per row, the prompt kernel
FORMS = [(3, 300, 0), (3, 1200, 0), (200, 300, 0), (70, 1200, 0), (2, 300, 40)]


def _attend(ops, form, q, k, v, sinks):
    B, n, T = form
    n_q, D = q.shape[-2:]
    cache = ops.KVCache(B, k.shape[2], D, (n + 63) // 64 * 64)
    cache.write(k, v)
    if T:
        return ops.AttnPrefill(B, T, n_q, k.shape[2], D, n).forward(q, cache, pos0=n - T, sinks=sinks)
    lens = torch.full((B,), n, dtype=torch.int32, device="cuda")
    return ops.AttnDecode(B, n_q, k.shape[2], D, n).forward(q, cache, lens, sinks)


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_scores_of_any_size(ops, form, D, sign):
    """Scores of about +-2^34 and 2^60 in powers of two, one of them larger than the others by a tenth: it takes all."""
    B, n, T = form
    n_q, n_kv = 16, 8
    g = torch.Generator(device="cuda").manual_seed(D)
    direction = torch.randn(D, generator=g, device="cuda").sign()
    for size in (2.0 ** 34, 2.0 ** 60):
        q = (direction * sign * size / math.sqrt(D)).expand(*((B, T) if T else (B,)), n_q, D).contiguous()
        level = 1.0 + 0.5 * torch.rand(B, n, n_kv, 1, generator=g, device="cuda")
        best = torch.randint(0, n - T if T else n, (B, n_kv), generator=g, device="cuda")
        level.scatter_(1, best[:, None, :, None], 1.75 if sign > 0 else 0.75)
        k = (level * direction).bfloat16()
        v = torch.randn(B, n, n_kv, D, generator=g, device="cuda").bfloat16()
        got = _attend(ops, form, q, k, v, None)
        want = v.gather(1, best[:, None, :, None].expand(B, 1, n_kv, D)).squeeze(1).repeat_interleave(n_q // n_kv, 1)
        want = want[:, None].expand_as(got) if T else want
        assert torch.equal(got, want), size


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("D", [32, 64])
def test_a_sink_far_above_every_score(ops, form, D):
    """The sink lies 125 to 145 powers of two above the scores, which are all equal: what is left is the mean of the values
    times 2^-shift, of values large enough for bf16 to hold it."""
    B, n, T = form
    n_q, n_kv = 16, 8
    g = torch.Generator(device="cuda").manual_seed(D)
    q = torch.zeros(*((B, T) if T else (B,)), n_q, D, device="cuda")
    k = torch.randn(B, n, n_kv, D, generator=g, device="cuda").bfloat16()
    v = (2.0 ** 40 * (1 + torch.rand(B, n, n_kv, D, generator=g, device="cuda"))).bfloat16()
    shift = torch.linspace(125, 145, n_q, device="cuda")
    sinks = shift * math.log(2.0)
    shift = sinks.double() / math.log(2.0)
    got = _attend(ops, form, q, k, v, sinks).double()
    seen = torch.arange(n - T + 1, n + 1, device="cuda") if T else torch.tensor([n], device="cuda")
    total = v.double().cumsum(1)[:, seen - 1]                                        # [B, T or 1, n_kv, D]
    want = total.repeat_interleave(n_q // n_kv, 2) * torch.exp2(-shift)[:, None]
    want = want if T else want[:, 0]
    # bf16: 2^-9; the exponent as a float near 145: 2^-17; its factor near 2^-145 has 2^-5 of itself as its last bit
    assert bool(((got - want).abs() <= want * (2.0 ** -8 + torch.exp2(shift - 149)[:, None])).all())


@pytest.mark.parametrize("form", FORMS + [(1, 300, 300)])
@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("step", [-12.0, 0.0, 3.0, 7.75, 8.25, 40.0])
def test_scores_that_climb_from_block_to_block(ops, form, D, step):
    """The largest score of a 64-slot block is `step` powers of two above the block before: references that stay, that are
    raised in every block, and in every second or third one.  And a row alone has the bits it has in any other form."""
    B, n, T = form
    n_q, n_kv = 16, 8
    g = torch.Generator(device="cuda").manual_seed(int(step * 4) + D)
    direction = torch.randn(D, generator=g, device="cuda").sign()
    q = direction.expand(*((B, T) if T else (B,)), n_q, D) / math.log2(math.e) / math.sqrt(D)
    level = (torch.arange(n, device="cuda") // 64 * step)[None, :, None, None] - 2 * torch.rand(B, n, n_kv, 1, generator=g, device="cuda")
    k = (level * direction).bfloat16()                      # scores: about `level` powers of two
    v = torch.randn(B, n, n_kv, D, generator=g, device="cuda").bfloat16()
    sinks = torch.randn(n_q, generator=g, device="cuda")
    got = _attend(ops, form, q.contiguous(), k, v, sinks)
    rows = got[:, -1] if T else got                         # the last position sees everything
    s = (q[:, -1] if T else q).double().view(B, n_kv, 2, D) @ k.double().permute(0, 2, 3, 1) / math.sqrt(D)
    w = torch.softmax(torch.cat([s, sinks.double().view(1, n_kv, 2, 1).expand(B, -1, -1, 1)], -1), -1)[..., :-1]
    want = (w @ v.double().transpose(1, 2)).view(B, n_q, D)
    size = (w @ v.double().abs().transpose(1, 2)).view(B, n_q, D)
    # bf16: 2^-9 of the result; scores of up to 2^8 in fp32, and their sums: 2^-15; weights and queries of 16 bits: 2^-15
    assert bool(((rows.double() - want).abs() <= want.abs() * 2.0 ** -8 + size * 2.0 ** -13).all())
    if n <= 512:
        assert torch.equal(rows[:1], _attend(ops, (1, n, 0), (q[:1, -1] if T else q[:1]).contiguous(), k[:1], v[:1], sinks))


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("longest", [1000, 2000, 3500, 7000, 16500])   # room for up to 3, 4, 7, 14 and 33 chunks of 512 positions
def test_rows_of_few_chunks_where_the_launch_has_room_for_many(ops, longest, D):
    """The partials of chunks that a row does not have are never written: whatever lies there does not reach its result,
    and neither does how many of them there are."""
    lens = [n for c in (0, 1, 2, 3, 4, 7, 8, 9, 15, 16, 17, 32) for n in (512 * c, 512 * c + 1) if n <= longest] + [longest]
    B, n_q, n_kv = len(lens), 16, 2
    g = torch.Generator(device="cuda").manual_seed(longest + D)
    q = torch.randn(B, n_q, D, generator=g, device="cuda")
    k, v = (torch.randn(B, longest, n_kv, D, generator=g, device="cuda").bfloat16() for _ in range(2))
    sinks = torch.randn(n_q, generator=g, device="cuda")
    cache = ops.KVCache(B, n_kv, D, (longest + 63) // 64 * 64)
    cache.write(k, v)
    attn = ops.AttnDecode(B, n_q, n_kv, D, longest)
    attn.ws.fill_(0xFF)   # NaN
    got = attn.forward(q, cache, torch.tensor(lens, dtype=torch.int32, device="cuda"), sinks)
    for b, n in enumerate(lens):
        s = q[b].double().view(n_kv, n_q // n_kv, D) @ k[b, :n].double().permute(1, 2, 0) / math.sqrt(D)
        w = torch.softmax(torch.cat([s, sinks.double().view(n_kv, -1, 1)], -1), -1)[..., :-1]
        want, size = ((w @ x.double().transpose(0, 1)).view(n_q, D) for x in (v[b, :n], v[b, :n].abs()))
        # bf16: 2^-9 of the result; weights and queries of 16 bits, scores and sums in fp32: 2^-14
        assert bool(((got[b].double() - want).abs() <= want.abs() * 2.0 ** -8 + size * 2.0 ** -13).all()), n
