"""GPU parity of the MoE path against the CPU oracle, through the C ABI."""
import ctypes as C

import numpy as np
import pytest
import torch

from conftest import TOL_MAX, TOL_MEAN, rel_errors

pytestmark = pytest.mark.gpu


def _bf16(t):
    return t.to(torch.bfloat16)


def _rand_layer(E, H, I, seed, std=0.02, dev="cuda"):
    g = torch.Generator(device="cpu").manual_seed(seed)
    def n(*shape, s=std):
        return _bf16(torch.randn(*shape, generator=g) * s)
    return dict(w_router=n(E, H), b_router=n(E), w1=n(E, 2 * I, H), b1=n(E, 2 * I),
                w2=n(E, H, I), b2=n(E, H))


def _f32np(t):
    return t.float().cpu().numpy()


# ---------------------------------------------------------------- routing: bit-exact integers
@pytest.mark.parametrize("B,E,k", [(1, 8, 4), (7, 8, 4), (64, 32, 4), (1024, 32, 4), (333, 128, 4),
                                   (4096, 128, 4), (100, 256, 8), (65, 40, 3), (0, 32, 4)])
def test_route_matches_oracle(ops, orc, B, E, k):
    rng = np.random.default_rng(1000 + B + E)
    logits = rng.standard_normal((B, E)).astype(np.float32)
    tw, ti, off, srt, inv, tiles = ops.moe_route(torch.from_numpy(logits).cuda(), k, rows_per_tile=128)
    torch.cuda.synchronize()
    if B == 0:
        assert off.cpu().numpy().tolist() == [0] * (E + 1)
        assert int(tiles[0]) == 0
        return
    ov, oi = orc.topk_softmax(logits, k)
    ooff, osrt, oinv = orc.group(oi, E)
    np.testing.assert_array_equal(ti.cpu().numpy(), oi)
    np.testing.assert_array_equal(off.cpu().numpy(), ooff)
    np.testing.assert_array_equal(srt.cpu().numpy(), osrt)
    np.testing.assert_array_equal(inv.cpu().numpy(), oinv)
    np.testing.assert_allclose(tw.cpu().numpy(), ov, rtol=2e-6, atol=1e-7)
    # tile list: every expert's rows cut into tiles of 128, in expert order
    t = tiles.cpu().numpy()
    exp = []
    for e in range(E):
        r0, r1 = int(ooff[e]), int(ooff[e + 1])
        for s in range(r0, r1, 128):
            exp.append((e, s, min(128, r1 - s)))
    assert t[0] == len(exp)
    assert [tuple(x) for x in t[1:1 + 3 * len(exp)].reshape(-1, 3)] == exp


def test_route_ties_lowest_expert_first(ops, orc):
    logits = np.zeros((5, 32), np.float32)
    logits[1, [3, 9, 20, 31]] = 1.0
    logits[2, :] = np.arange(32) % 4            # many equal values
    logits[3, 7] = -np.inf
    logits[4, :] = -1.0
    logits[4, [30, 2]] = 5.0
    tw, ti, off, srt, inv, _ = ops.moe_route(torch.from_numpy(logits).cuda(), 4)
    ov, oi = orc.topk_softmax(logits, 4)
    np.testing.assert_array_equal(ti.cpu().numpy(), oi)
    assert ti.cpu().numpy()[0].tolist() == [0, 1, 2, 3]
    assert ti.cpu().numpy()[1].tolist() == [3, 9, 20, 31]
    assert ti.cpu().numpy()[4].tolist()[:2] == [2, 30]
    np.testing.assert_allclose(tw.cpu().numpy(), ov, rtol=2e-6)


def test_route_skewed_all_to_one_expert(ops, orc):
    B, E, k = 2048, 32, 4
    logits = np.random.default_rng(5).standard_normal((B, E)).astype(np.float32)
    logits[:, 5] += 100.0
    logits[:, 17] += 50.0
    tw, ti, off, srt, inv, _ = ops.moe_route(torch.from_numpy(logits).cuda(), k)
    ov, oi = orc.topk_softmax(logits, k)
    ooff, osrt, oinv = orc.group(oi, E)
    np.testing.assert_array_equal(off.cpu().numpy(), ooff)
    np.testing.assert_array_equal(srt.cpu().numpy(), osrt)
    np.testing.assert_array_equal(inv.cpu().numpy(), oinv)


# ---------------------------------------------------------------- router GEMM
@pytest.mark.parametrize("B,H,E", [(1, 256, 8), (37, 256, 8), (1024, 2880, 32), (100, 2880, 128)])
def test_router_gemm(ops, B, H, E):
    g = torch.Generator().manual_seed(B + E)
    t = _bf16(torch.randn(B, H, generator=g)).cuda()
    w = _bf16(torch.randn(E, H, generator=g) * 0.02).cuda()
    b = _bf16(torch.randn(E, generator=g) * 0.02).float().cuda()
    got = ops.router_gemm(t, w, b).cpu().numpy()
    want = (t.double().cpu() @ w.double().cpu().T + b.double().cpu()).numpy()
    assert np.abs(got - want).max() <= 1e-4 * max(1.0, np.abs(want).max())


@pytest.mark.parametrize("E", [1, 17, 33, 65, 129, 255])    # blocks of 16 experts, whole and not, in one to four parts of a stage
@pytest.mark.parametrize("H", [32, 224, 256, 288, 768])     # stages of 256 inputs: a piece of one, one, one and a piece, three
def test_router_stages(ops, E, H):
    g = torch.Generator(device="cuda").manual_seed(E + H)
    n = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    t, w, b = n(21, H), n(E, H), n(E).float()
    want = t.double() @ w.double().T + b.double()
    for tokens in (1, 5, 16, 21):
        got = ops.router_gemm(t[:tokens].contiguous(), w, b)
        # as in test_router_rows_are_the_same_in_groups_of_any_size
        assert bool(((got.double() - want[:tokens]).abs() <= 2.0 ** -24 * (H / 8 + 8) * 8 * H ** 0.5).all()), tokens


@pytest.mark.parametrize("E", [32, 33, 48, 65, 129, 255])   # blocks of 16 experts, whole and not, in one to four parts of a stage
@pytest.mark.parametrize("H", [32, 96, 256, 288, 768, 2912])
def test_router_logits_of_shared_experts_and_of_all_in_one_workgroup(ops, E, H):
    """Without the gating, more than 32 experts are shared out up to 1024 tokens; 1025 have all experts in a workgroup.  Same bits."""
    g = torch.Generator(device="cuda").manual_seed(E * H)
    n = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    t, w, b = n(1025, H), n(E, H), n(E).float()
    want = t.double() @ w.double().T + b.double()
    whole = ops.router_gemm(t, w, b)
    # as in test_router_rows_are_the_same_in_groups_of_any_size
    assert bool(((whole.double() - want).abs() <= 2.0 ** -24 * (H / 8 + 8) * 8 * H ** 0.5).all())
    for tokens in (1, 17, 511, 1024):
        assert torch.equal(ops.router_gemm(t[:tokens].contiguous(), w, b), whole[:tokens]), tokens


# the last experts' rows, and the last tokens' too, begin 4 GiB and more behind the first one
@pytest.mark.parametrize("B,H,E", [(3, 8421536, 256), (4, 715827904, 4), (3, 69273696, 32)])
def test_router_matrices_of_more_than_four_gib(ops, B, H, E):
    g = torch.Generator(device="cuda").manual_seed(E)
    t = torch.zeros(B, H, dtype=torch.bfloat16, device="cuda")
    w = torch.zeros(E, H, dtype=torch.bfloat16, device="cuda")
    at = torch.tensor([0, 8, 255, 256, 1000, H // 2, H - 300, H - 33, H - 1], device="cuda")
    t[:, at] = torch.randint(-3, 4, (B, len(at)), generator=g, device="cuda").bfloat16()
    w[:, at] = torch.randint(-9, 10, (E, len(at)), generator=g, device="cuda").bfloat16()
    b = torch.arange(E, device="cuda").float()
    assert (E - 1) * H * 2 >= 2 ** 32 and H % 32 == 0
    got = ops.router_gemm(t, w, b)
    want = (t[:, at].float() @ w[:, at].float().T) + b      # whole numbers, exact in any order
    assert torch.equal(got, want)


# ---------------------------------------------------------------- weight packing
@pytest.mark.parametrize("E", [32, 64, 128, 256])           # a stage in one part, one, two and four
@pytest.mark.parametrize("H", [32, 320, 1792, 2048, 2080, 3104])   # one k-step in all; whole stages of 256 inputs, and a last one of one k-step or two
def test_router_rows_are_the_same_in_groups_of_any_size(ops, E, H):
    """Workgroups of 4, 8 and 16 token rows: up to 1024 tokens, 2048, more."""
    g = torch.Generator(device="cuda").manual_seed(E + H)
    n = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    t, w, b = n(4099, H), n(E, H), n(E).float()
    want = t.double() @ w.double().T + b.double()
    for tokens in (1024, 1025, 2048, 2049, 4096, 4099):
        got = ops.router_gemm(t[:tokens], w, b)
        # exact products, fp32 sums of H of them: 2^-24 for each of at most H / 8 + 8 roundings, sizes of about sqrt(H)
        assert bool(((got.double() - want[:tokens]).abs() <= 2.0 ** -24 * (H / 8 + 8) * 8 * H ** 0.5).all()), tokens
        assert torch.equal(got[-3:], ops.router_gemm(t[tokens - 3:tokens], w, b)), tokens


def test_pack_weight_layout(ops):
    n_mat, N, K = 2, 128, 128
    w = torch.arange(n_mat * N * K, dtype=torch.float32).reshape(n_mat, N, K) % 251
    wp = ops.pack_weight(w.to(torch.bfloat16).cuda()).float().cpu().numpy().reshape(n_mat, N // 32, K // 16, 64, 8)
    wp32 = ops.pack_weight(w.cuda()).float().cpu().numpy().reshape(n_mat, N // 32, K // 16, 64, 8)
    wn = w.numpy()
    for m, nb, ks, lane in [(0, 0, 0, 0), (1, 3, 7, 63), (0, 2, 5, 33), (1, 1, 1, 31)]:
        row, k0 = nb * 32 + lane % 32, ks * 16 + (lane // 32) * 8
        np.testing.assert_array_equal(wp[m, nb, ks, lane], wn[m, row, k0:k0 + 8])
        np.testing.assert_array_equal(wp32[m, nb, ks, lane], wn[m, row, k0:k0 + 8])
    # GLU pairing: virtual row v of a 32-row block -> pair (v//32)*16 + v%16, 16 gates then 16 ups
    wg = ops.pack_weight(w.to(torch.bfloat16).cuda(), glu=True).float().cpu().numpy().reshape(n_mat, N // 32, K // 16, 64, 8)
    for m, nb, ks, lane in [(0, 0, 0, 0), (0, 1, 2, 5), (1, 3, 7, 63), (1, 2, 0, 40)]:
        v = nb * 32 + lane % 32
        row = 2 * ((v // 32) * 16 + v % 16) + (v // 16) % 2
        k0 = ks * 16 + (lane // 32) * 8
        np.testing.assert_array_equal(wg[m, nb, ks, lane], wn[m, row, k0:k0 + 8])


# ---------------------------------------------------------------- whole MoE block vs oracle
@pytest.mark.parametrize("B,E,H,I,seed", [
    (8, 8, 256, 256, 1),        # tiny-model shape, decode batch
    (1, 8, 256, 256, 2),
    (96, 8, 256, 256, 3),       # 48 rows per expert
    (300, 8, 256, 256, 4),      # >128 rows per expert: 256-row tiles
    (700, 8, 256, 256, 5),      # >256 rows per expert: several tiles per expert
    (64, 32, 2880, 2880, 6),    # 20B shape, few tokens
])
def test_moe_forward_matches_oracle(ops, orc, B, E, H, I, seed):
    L = _rand_layer(E, H, I, seed)
    g = torch.Generator().manual_seed(100 + seed)
    t = _bf16(torch.randn(B, H, generator=g))
    layer = ops.MoeLayer(*[L[n].cuda() for n in ("w_router", "b_router", "w1", "b1", "w2", "b2")],
                         max_tokens=max(B, 1))
    out = layer.forward(t.cuda())
    torch.cuda.synchronize()
    logits, tw, ti, off, srt, inv = [x.cpu().numpy() for x in layer.routing_views()]
    want, ologits, otv, oti = orc.moe_layer(_f32np(t), *[_f32np(L[n]) for n in
                                            ("w_router", "b_router", "w1", "b1", "w2", "b2")],
                                            k=4, limit=7.0, stage=orc.STAGE_SWIGLU, want_routing=True)
    np.testing.assert_allclose(logits, ologits, atol=2e-5 * max(1.0, np.abs(ologits).max()))
    # grouping is bit-exact given the GPU's own logits
    ov, oi = orc.topk_softmax(logits, 4)
    ooff, osrt, oinv = orc.group(oi, E)
    np.testing.assert_array_equal(ti, oi)
    np.testing.assert_array_equal(off, ooff)
    np.testing.assert_array_equal(srt, osrt)
    np.testing.assert_array_equal(inv, oinv)
    # rows whose GPU routing equals the oracle's routing (ties in the 1e-6 range may differ)
    same = (oti == ti).all(axis=1)
    assert same.mean() > 0.98
    mx, mean = rel_errors(out.cpu().numpy()[same], want[same])
    assert mx <= TOL_MAX and mean <= TOL_MEAN, (mx, mean)


def test_moe_forward_accumulate_and_determinism(ops):
    E, H, I, B = 8, 256, 256, 200
    L = _rand_layer(E, H, I, 9)
    t = _bf16(torch.randn(B, H, generator=torch.Generator().manual_seed(3))).cuda()
    layer = ops.MoeLayer(*[L[n].cuda() for n in ("w_router", "b_router", "w1", "b1", "w2", "b2")],
                         max_tokens=B)
    a = layer.forward(t).clone()
    b = layer.forward(t).clone()
    assert torch.equal(a, b)                      # run-to-run bit reproducible
    x = torch.randn(B, H, device="cuda")
    y = x.clone()
    layer.forward(t, out=y, accumulate=True)
    assert torch.equal(y, x + a)


@pytest.mark.parametrize("B,E,H,I", [(3000, 16, 256, 512), (1500, 64, 512, 256)])
def test_moe_forward_skewed_routing_is_batch_invariant(ops, orc, B, E, H, I):
    """Zipf-skewed routing (experts with many row tiles next to experts with a few rows): the work
    list is then cut into per-XCD parts by estimated cost, with cuts that fall inside tiles.  Every
    token's output must not depend on what else is in the batch: the full batch equals, bit for bit,
    the same tokens run in two halves (other tiles, other cuts), and a sample equals the oracle."""
    L = _rand_layer(E, H, I, 21)
    ranks = np.random.default_rng(B).permutation(E) + 1
    L["b_router"] = torch.from_numpy((1.5 * np.log(1.0 / ranks ** 1.1)).astype(np.float32))
    g = torch.Generator().manual_seed(B)
    t = _bf16(torch.randn(B, H, generator=g))
    layer = ops.MoeLayer(*[L[n].cuda() for n in ("w_router", "b_router", "w1", "b1", "w2", "b2")],
                         max_tokens=B)
    full = layer.forward(t.cuda()).clone()
    logits, tw, ti, off, srt, inv = [x.cpu().numpy() for x in layer.routing_views()]
    counts = np.diff(off)
    assert counts.max() >= 4 * counts.mean() and counts.max() > 3 * 160   # several tiles for one expert
    h = B // 2 + 7
    first = layer.forward(t[:h].cuda()).clone()
    second = layer.forward(t[h:].cuda()).clone()
    assert torch.equal(full[:h], first)
    assert torch.equal(full[h:], second)
    n_chk = 40
    want, _, _, oti = orc.moe_layer(_f32np(t)[:n_chk], *[_f32np(L[n]) for n in
                                    ("w_router", "b_router", "w1", "b1", "w2", "b2")],
                                    k=4, limit=7.0, stage=orc.STAGE_SWIGLU, want_routing=True)
    same = (oti == ti[:n_chk]).all(axis=1)
    assert same.mean() > 0.9
    mx, mean = rel_errors(full.cpu().numpy()[:n_chk][same], want[same])
    assert mx <= TOL_MAX and mean <= TOL_MEAN, (mx, mean)


# ---------------------------------------------------------------- SwiGLU epilogue and bias order, alone
def test_swiglu_special_cases_and_bias_order_through_a_one_expert_layer(ops, orc):
    """One expert, top-1, w2 = identity: the layer's output is the bf16-rounded clamped SwiGLU of
    chosen (gate, up) values plus b2, so the epilogue of GEMM1 (run.cpp:669-686: gate = min(g, 7),
    up = clamp(u, -7, 7), g * sigmoid(1.702 g) * (up + 1)), the (gate, up) interleave of mlp1's rows
    and the order of both bias vectors are checked on their own, special cases included:
    g > 7, u > 7, u < -7 (up + 1 = -6), g -> -inf (0)."""
    H = I = 64
    B = 4
    gv = np.array([8.0, 7.0, 6.5, -100.0, 0.5, -0.5, 30.0, -8.0], np.float32)
    uv = np.array([-8.0, 8.0, 0.25, 7.0, -7.0, -6.5, 100.0, -1.0], np.float32)
    j = np.arange(I)
    g_j, u_j = gv[j % 8], uv[(j // 8) % 8]
    w1 = np.zeros((1, 2 * I, H), np.float32)
    w1[0, 0::2, 0] = g_j                       # row 2j = gate of pair j, row 2j+1 = its up
    w1[0, 1::2, 0] = u_j
    b1 = np.zeros((1, 2 * I), np.float32)
    b1[0, 0::2] = 0.125 * (j % 3)
    b1[0, 1::2] = -0.25 * (j % 5)
    b2 = (0.5 * (j % 7) - 1.0).astype(np.float32)[None]
    w2 = np.eye(H, I, dtype=np.float32)[None]
    s = np.array([1.0, 0.5, -1.0, 2.0], np.float32)
    t = np.zeros((B, H), np.float32)
    t[:, 0] = s
    t[:, 5] = 3.0                              # a column no weight reads
    tt = lambda a: torch.from_numpy(a).to(torch.bfloat16).cuda()
    mk = lambda bias2: ops.MoeLayer(torch.zeros(1, H, dtype=torch.bfloat16).cuda(), torch.zeros(1).cuda(), tt(w1),
                                    torch.from_numpy(b1).cuda(), tt(w2), torch.from_numpy(bias2).cuda(), top_k=1,
                                    max_tokens=B)
    got = mk(np.zeros_like(b2)).forward(tt(t)).cpu().numpy()
    with_b2 = mk(b2).forward(tt(t)).cpu().numpy()
    np.testing.assert_allclose(with_b2 - got, np.broadcast_to(b2, got.shape), atol=1e-5)   # b2[j] lands on column j
    gate = s[:, None] * g_j[None, :] + b1[0, 0::2][None, :]
    up = s[:, None] * u_j[None, :] + b1[0, 1::2][None, :]
    pre = np.empty((B, 2 * I), np.float32)
    pre[:, 0::2], pre[:, 1::2] = gate, up
    want = orc.swiglu(pre, 7.0)
    # closed form in float64, independent of the oracle
    gc_, uc_ = np.minimum(gate.astype(np.float64), 7.0), np.clip(up.astype(np.float64), -7.0, 7.0)
    closed = gc_ / (1.0 + np.exp(-1.702 * gc_)) * (uc_ + 1.0)
    np.testing.assert_allclose(want, closed, rtol=1e-5, atol=1e-30)
    # the GPU result is bf16-rounded (2^-9 relative) after exp2/reciprocal of a few ulp
    np.testing.assert_allclose(got, closed, rtol=5e-3, atol=1e-30)
    # the special cases, by value
    big_g = gate > 7.0
    assert big_g.any() and (up < -7.0).any() and (up > 7.0).any() and (gate < -50).any()
    sig7 = 7.0 / (1.0 + np.exp(-1.702 * 7.0))
    np.testing.assert_allclose(got[big_g], (sig7 * (uc_ + 1.0))[big_g], rtol=5e-3)
    np.testing.assert_allclose(got[big_g & (up < -7.0)], sig7 * -6.0, rtol=5e-3)
    assert (got[gate < -50] == 0).all()


@pytest.mark.parametrize("B,E,k,skew", [(2048, 8, 4, 0.0), (2300, 40, 4, 2.0), (4096, 128, 4, 3.0), (3000, 256, 8, 0.0),
                                        (9000, 32, 1, 1.0)])
def test_grouping_by_many_workgroups(ops, orc, B, E, k, skew):
    """From 8192 (token, expert) pairs on, the layer sorts them with one workgroup per 1024 pairs
    (counts per workgroup, then offsets + scatter) instead of a single workgroup: offsets,
    permutation and inverse must still be the stable counting sort, bit for bit, and the layer
    output (which follows the tile list the same kernels write) must match the oracle."""
    H = I = 64
    g = torch.Generator().manual_seed(B + E)
    n = lambda *s: _bf16(torch.randn(*s, generator=g) * 0.05)
    br = _bf16(n(E).float() - skew * torch.arange(E) / E)
    L = dict(w_router=n(E, H), b_router=br, w1=n(E, 2 * I, H), b1=n(E, 2 * I), w2=n(E, H, I), b2=n(E, H))
    names = ("w_router", "b_router", "w1", "b1", "w2", "b2")
    t = _bf16(torch.randn(B, H, generator=g))
    layer = ops.MoeLayer(*[L[x].cuda() for x in names], top_k=k, max_tokens=B)
    out = layer.forward(t.cuda())
    torch.cuda.synchronize()
    logits, tw, ti, off, srt, inv = [x.cpu().numpy() for x in layer.routing_views()]
    assert B * k >= 8192
    _, oi = orc.topk_softmax(logits, k)
    ooff, osrt, oinv = orc.group(oi, E)
    np.testing.assert_array_equal(ti, oi)
    np.testing.assert_array_equal(off, ooff)
    np.testing.assert_array_equal(srt, osrt)
    np.testing.assert_array_equal(inv, oinv)
    want, _, _, oti = orc.moe_layer(_f32np(t), *[_f32np(L[x]) for x in names], k=k, limit=7.0,
                                    stage=orc.STAGE_SWIGLU, want_routing=True)
    same = (oti == ti).all(axis=1)
    assert same.mean() > 0.95
    mx, mean = rel_errors(out.cpu().numpy()[same], want[same])
    assert mx <= TOL_MAX and mean <= TOL_MEAN, (mx, mean)


# ---------------------------------------------------------------- prompt-pass sizes: 256-row tiles
@pytest.mark.parametrize("B,E,H,I,skew", [
    (2100, 8, 320, 320, 0.0),      # K = 320: ten stages; N = 640 and 320: a partial column tile each
    (2600, 16, 256, 512, 1.1),     # skewed: experts of many tiles beside experts of a few rows
    (1300, 4, 512, 256, 0.0),      # an expert's last tile of a few rows
    (4100, 32, 2880, 2880, 0.0),   # the 20B layer at 4100 tokens
])
def test_moe_forward_of_a_prompt_pass_equals_the_same_tokens_in_small_batches(ops, orc, B, E, H, I, skew):
    """From 512 rows per expert on average the block runs kernels of their own (256-row tiles, both
    operands through LDS).  They must give every token the bits that the streaming kernels give it:
    the full batch equals the same tokens run in batches of 1/8 of the size, and a sample equals the oracle."""
    L = _rand_layer(E, H, I, 31)
    if skew:
        ranks = np.random.default_rng(B).permutation(E) + 1
        L["b_router"] = torch.from_numpy((1.5 * np.log(1.0 / ranks ** skew)).astype(np.float32))
    t = _bf16(torch.randn(B, H, generator=torch.Generator().manual_seed(B)))
    layer = ops.MoeLayer(*[L[n].cuda() for n in ("w_router", "b_router", "w1", "b1", "w2", "b2")],
                         max_tokens=B)
    assert B * 4 >= 512 * E
    full = layer.forward(t.cuda()).clone()
    ti = layer.routing_views()[2].cpu().numpy()
    step = B // 8 + 3
    assert step * 4 < 512 * E
    for r0 in range(0, B, step):
        part = layer.forward(t[r0:r0 + step].cuda())
        assert torch.equal(full[r0:r0 + step], part), r0
    n_chk = 24
    rows = np.r_[0:n_chk // 2, B - n_chk // 2:B]
    want, _, _, oti = orc.moe_layer(_f32np(t)[rows], *[_f32np(L[n]) for n in
                                    ("w_router", "b_router", "w1", "b1", "w2", "b2")],
                                    k=4, limit=7.0, stage=orc.STAGE_SWIGLU, want_routing=True)
    same = (oti == ti[rows]).all(axis=1)
    assert same.mean() > 0.9
    mx, mean = rel_errors(full.cpu().numpy()[rows][same], want[same])
    assert mx <= TOL_MAX and mean <= TOL_MEAN, (mx, mean)


# k: one of four places, three, all four, five of eight places, all eight; H: a piece of a thread's chunk, one chunk, the next
# remainder, three chunks short of the end and whole, a loop
@pytest.mark.parametrize("k", [1, 3, 4, 5, 8])
@pytest.mark.parametrize("H", [64, 1024, 1088, 2880, 3072, 4096])
def test_combine_adds_every_product_in_expert_order(ops, k, H):
    """With a second product of zeros an expert's row is its bias: what is left is the rounding of at most k products and k
    sums."""
    E, B = 16, 19
    g = torch.Generator(device="cuda").manual_seed(k * H)
    n = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    layer = ops.MoeLayer(n(E, H), n(E), n(E, 128, H), n(E, 128), torch.zeros(E, H, 64, device="cuda").bfloat16(), n(E, H),
                         top_k=k, max_tokens=64)
    t, out = n(B, H), torch.randn(B, H, generator=g, device="cuda")
    before = out.clone()
    layer.forward(t, out=out, accumulate=True)
    fresh = layer.forward(t)
    _, w, ids = layer.routing_views()[:3]
    ids, order = ids.long().sort(dim=1)
    w = w.gather(1, order)
    terms = torch.stack([layer.b2[ids[:, s]].double() * w[:, s, None].double() for s in range(k)])
    bound = 2 * k * 2.0 ** -24 * terms.abs().sum(0)
    assert bool(((fresh - terms.sum(0)).abs() <= bound).all())
    assert torch.equal(out, before + fresh)


@pytest.mark.parametrize("E,k", [(4, 4), (32, 4), (40, 3), (256, 8)])
def test_routing_of_rows_that_are_no_numbers(ops, orc, E, k):
    """Rows of NaN, a row with one, and one of which only k - 1 values are numbers: k different experts each, weights of NaN
    where a NaN is picked; the rows between them as if they were alone."""
    B = 12
    logits = np.random.default_rng(E).standard_normal((B, E)).astype(np.float32)
    logits[[0, 7]] = np.nan
    logits[3, E // 2] = np.nan
    logits[5, k - 1:] = np.nan
    tw, ti, off, srt, inv, _ = [x.cpu().numpy() if x is not None else None for x in ops.moe_route(torch.from_numpy(logits).cuda(), k)]
    ranked = np.where(np.isnan(logits), -np.inf, logits).astype(np.float32)
    ov, oi = orc.topk_softmax(ranked, k)
    np.testing.assert_array_equal(ti, oi)
    picked_nan = np.isnan(np.take_along_axis(logits, oi.astype(np.int64), axis=1)).any(axis=1)
    assert np.isnan(tw[picked_nan]).all()
    np.testing.assert_allclose(tw[~picked_nan], ov[~picked_nan], rtol=2e-6, atol=1e-7)
    for got, want in zip((off, srt, inv), orc.group(oi, E)):
        np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("B", [3, 16, 17, 100])       # grouped by the router's own workgroup, and by a kernel behind it
@pytest.mark.parametrize("E", [4, 32, 128])
def test_tokens_that_are_no_numbers_leave_the_others_alone(ops, B, E):
    g = torch.Generator(device="cuda").manual_seed(B + E)
    n = lambda *s, std=1.0: (torch.randn(*s, generator=g, device="cuda") * std).bfloat16()
    H = I = 128
    layer = ops.MoeLayer(n(E, H, std=0.1), n(E), n(E, 2 * I, H, std=0.1), n(E, 2 * I), n(E, H, I, std=0.1), n(E, H), top_k=4,
                         max_tokens=128)
    t = n(B, H)
    want = layer.forward(t).clone()
    bad = list(range(0, B, 2)) if B <= 16 else list(range(0, B, 7))
    broken = t.clone()
    broken[bad] = float("nan")
    got = layer.forward(broken)
    rest = [b for b in range(B) if b not in bad]
    assert bool(torch.isnan(got[bad]).all())
    assert torch.equal(got[rest], want[rest])


@pytest.mark.parametrize("E", [1, 2, 31, 32, 33, 64, 65, 129, 256])   # one to eight experts per lane, lanes without one
@pytest.mark.parametrize("k", [1, 2, 4, 7, 8])
def test_routing_of_equal_and_infinite_logits(ops, E, k):
    """Few different values, zeros of both signs and -infinity among them: the picks are the first k by value, then by expert;
    the weights are within the rounding of an exponential, a sum of k and a division in fp32."""
    if k > E:
        pytest.skip("more picks than experts")
    rng = np.random.default_rng(E * 8 + k)
    logits = rng.choice(np.array([-np.inf, -3.5, -0.0, 0.0, 1.25, 1.25, 2.0], np.float32), size=(67, E))
    logits[:, rng.integers(E)] = 2.0                    # a largest value that is a number
    tw, ti = [x.cpu().numpy() for x in ops.moe_route(torch.from_numpy(logits).cuda(), k)[:2]]
    want = np.argsort(-(logits + np.float32(0)), axis=1, kind="stable")[:, :k]
    np.testing.assert_array_equal(ti, want)
    picked = np.take_along_axis(logits, want, axis=1).astype(np.float64)
    e = np.exp(picked - picked[:, :1])
    np.testing.assert_allclose(tw, e / e.sum(1, keepdims=True), rtol=2e-6, atol=0)


@pytest.mark.parametrize("E", [33, 48, 64, 100, 128, 256])
@pytest.mark.parametrize("H", [64, 256, 2880])
def test_experts_shared_out_among_workgroups_score_and_gate_the_same(ops, E, H):
    """From 33 experts on (H = 256 and 64: from 129) up to 512 tokens have 16 experts per workgroup and are
    gated by another launch; 600 have one workgroup for all experts.  Same bits."""
    g = torch.Generator(device="cuda").manual_seed(E + H)
    n = lambda *s, std=1.0: (torch.randn(*s, generator=g, device="cuda") * std).bfloat16()
    layer = ops.MoeLayer(n(E, H, std=H ** -0.5), n(E).float(), n(E, 128, H, std=0.05), n(E, 128).float(), n(E, H, 64), n(E, H).float(),
                         top_k=4, max_tokens=600)
    t = n(600, H)
    out = layer.forward(t).clone()
    want = [v.clone() for v in layer.routing_views()[:3]]
    for tokens in (1, 3, 16, 17, 65, 256, 257, 512):
        got = layer.forward(t[:tokens].contiguous())
        for have, all_of_them in zip(layer.routing_views()[:3], want):
            assert torch.equal(have, all_of_them[:tokens]), tokens
        assert torch.equal(got, out[:tokens]), tokens


# 33 to 64 experts of more than 2048 inputs, up to 128 of 512 and more, beyond of any: shared out up to 512 tokens.  Up to 16
# tokens: partial products, unless 8 E floats are more than k H, three to seven tokens have fewer than 16 experts, or there are
# fewer than 256 inputs and 4096 weights
@pytest.mark.parametrize("H,E,tokens,router", [
    (4096, 32, 1, "parts"), (4096, 32, 17, "one"), (2112, 33, 1, "parts"), (2112, 33, 17, "shared"), (2112, 33, 513, "one"),
    (2048, 33, 17, "one"), (2048, 64, 16, "parts"), (2048, 64, 17, "one"), (512, 65, 16, "parts"), (512, 65, 17, "shared"),
    (448, 128, 17, "one"), (1088, 128, 512, "shared"), (1024, 128, 513, "one"), (576, 129, 512, "shared"), (576, 129, 513, "one"),
    (512, 256, 257, "shared"), (512, 256, 16, "parts"), (448, 256, 16, "shared"), (256, 64, 17, "one"), (192, 256, 17, "shared"),
    (128, 129, 512, "shared"), (128, 129, 513, "one"), (128, 128, 17, "one"), (64, 256, 1, "shared"), (192, 21, 1, "one"),
    (192, 22, 5, "parts"), (64, 64, 4, "one"), (256, 15, 2, "parts"), (256, 15, 7, "one"), (256, 15, 8, "parts"), (256, 16, 5, "parts")])
def test_which_calls_share_their_experts_out(ops, H, E, tokens, router):
    g = torch.Generator(device="cuda").manual_seed(H)
    n = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    layer = ops.MoeLayer(n(E, H), n(E).float(), n(E, 128, H), n(E, 128).float(), n(E, H, 64), n(E, H).float(), top_k=4, max_tokens=tokens)
    t = n(tokens, H)
    with ops.KernelTrace(16) as trace:
        layer.forward(t)
    launches = [name for name, _ in trace.results()]
    name = {"parts": "router_parts", "one": "router_gemm_topk", "shared": "router_gemm"}
    assert [x for x in launches if x.startswith("router")] == [name[router]]


# 48 experts of 768 x 2880: 1620 workgroups for one token, 3060 for two; 32 experts: any number
@pytest.mark.parametrize("E,tokens,by_one", [(48, 1, False), (48, 2, True), (32, 2, False)])
def test_two_tokens_over_more_workgroups_than_the_chip_holds_are_gated_by_one(ops, E, tokens, by_one):
    g = torch.Generator(device="cuda").manual_seed(E + tokens)
    n = lambda *s, std=1.0: (torch.randn(*s, generator=g, device="cuda") * std).bfloat16()
    H, I = 768, 2880
    layer = ops.MoeLayer(n(E, H, std=H ** -0.5), n(E).float(), n(E, 2 * I, H, std=0.05), n(E, 2 * I).float(), n(E, H, I, std=0.05),
                         n(E, H).float(), top_k=8, max_tokens=40)
    t = n(40, H)
    out = layer.forward(t).clone()
    with ops.KernelTrace(16) as trace:
        got = layer.forward(t[:tokens].contiguous())
    launches = [name for name, _ in trace.results()]
    assert "router_parts" in launches and ("topk_group" in launches) == by_one
    assert torch.equal(got, out[:tokens])


@pytest.mark.parametrize("E,H", [(49, 256), (64, 448), (65, 512), (128, 960), (129, 64), (129, 512), (256, 1984)])
def test_a_few_tokens_without_room_for_partial_products(ops, E, H):
    """One expert per token: 8 E floats are more than its row of the second product's output.  Up to 64 experts one workgroup does
    the whole routing, beyond the experts are shared out and one workgroup gates and groups the tokens; as in larger batches, to the bit."""
    g = torch.Generator(device="cuda").manual_seed(E + H)
    n = lambda *s, std=1.0: (torch.randn(*s, generator=g, device="cuda") * std).bfloat16()
    layer = ops.MoeLayer(n(E, H, std=H ** -0.5), n(E).float(), n(E, 128, H, std=0.05), n(E, 128).float(), n(E, H, 64), n(E, H).float(),
                         top_k=1, max_tokens=600)
    t = n(600, H)
    out = layer.forward(t).clone()
    want = [v.clone() for v in layer.routing_views()[:3]]
    for tokens in (1, 2, 3, 8, 15, 16):
        part = t[:tokens].contiguous()
        with ops.KernelTrace(16) as trace:
            got = layer.forward(part)
        launches = [name for name, _ in trace.results()]
        assert ("router_gemm" in launches and "topk_group" in launches) == (E > 64) and "router_parts" not in launches
        have = layer.routing_views()
        for a, b in zip(have, want):
            assert torch.equal(a, b[:tokens]), tokens
        for a, b in zip(have[3:], ops.moe_route(ops.router_gemm(part, layer.w_router, layer.b_router), 1)[2:5]):
            assert torch.equal(a, b), tokens
        assert torch.equal(got, out[:tokens]), tokens


# up to two tokens are gated by the workgroups of the first product, up to four with 16 to 32 experts (of 1280 inputs), up to 128
# experts; the others by one workgroup.  One expert per lane and four, lanes without one, one to 32 pairs
@pytest.mark.parametrize("mxfp4", [False, True])
@pytest.mark.parametrize("E,k", [(1, 1), (2, 2), (15, 8), (16, 1), (31, 5), (32, 8), (33, 4), (128, 8), (129, 8)])
def test_a_few_tokens_are_routed_as_in_any_batch(ops, E, k, mxfp4):
    g = torch.Generator(device="cuda").manual_seed(E * 9 + k)
    H, I = 1280, 192
    n = lambda *s, std=1.0: (torch.randn(*s, generator=g, device="cuda") * std).bfloat16()
    def matrix(rows, cols):
        if not mxfp4:
            return [n(E, rows, cols, std=0.05)]
        codes = torch.randint(0, 256, (E, rows, cols // 2), generator=g, device="cuda", dtype=torch.uint8)
        return [codes, torch.randint(118, 124, (E, rows, cols // 32), generator=g, device="cuda", dtype=torch.uint8)]
    bias = (torch.arange(E, device="cuda") % 3).float()   # a token of zeros: many equal logits
    layer = (ops.MoeLayerMxfp4 if mxfp4 else ops.MoeLayer)(
        n(E, H, std=H ** -0.5), bias, *matrix(2 * I, H), n(E, 2 * I).float(), *matrix(H, I), n(E, H).float(), top_k=k, max_tokens=40)
    t = n(40, H)
    t[2] = 0
    t[3] = float("nan")
    t[5] = 1e38           # products and sums that are infinite, or none
    same = lambda a, b: torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num())
    all_of_them = layer.forward(t).clone()
    for tokens in (1, 2, 3, 4, 5, 7, 8, 16):
        for first in (0, 2, 3, 4):
            part = t[first:first + tokens].contiguous()
            got = layer.forward(part)
            logits = ops.router_gemm(part, layer.w_router, layer.b_router)
            want = [logits, *ops.moe_route(logits, k)[:5]]
            for name, a, b in zip("logits weights ids offsets order place".split(), layer.routing_views(), want):
                assert same(a, b), (tokens, first, name)
            assert same(got, all_of_them[first:first + tokens]), (tokens, first)


@pytest.mark.parametrize("E,k", [(1, 1), (4, 4), (32, 4), (33, 8), (128, 4), (256, 8)])
def test_grouping_of_a_few_tokens_by_one_wave(ops, E, k):
    """gptoss::run_group, which has no C entry point, by its linker name, against gptoss_moe_route's kernels."""
    import ctypes as C
    from conftest import load_pkg
    lib = load_pkg("lib")
    f = getattr(lib.load(), "_ZN6gptoss9run_groupEiiiPfPiS1_S1_S1_S1_iS1_iP12ihipStream_tS1_")
    f.restype, f.argtypes = C.c_int, [C.c_int] * 3 + [C.c_void_p] * 6 + [C.c_int, C.c_void_p, C.c_int, C.c_void_p, C.c_void_p]
    g = torch.Generator(device="cuda").manual_seed(E + k)
    for tokens in (1, 2, 5, 15, 16, 17):
        logits = torch.randn(tokens, E, generator=g, device="cuda")
        w, i, off, srt, inv, tiles = ops.moe_route(logits, k, rows_per_tile=32)
        got = [torch.full_like(x, -1) for x in (off, srt, inv, tiles)]
        bounds = torch.full((16 + tokens * k + E,), -1, dtype=torch.int32, device="cuda")
        lib.check(f(tokens, E, k, w.data_ptr(), i.data_ptr(), *[x.data_ptr() for x in got], 32, bounds.data_ptr(), 32,
                    torch.cuda.current_stream().cuda_stream, None))
        n_tiles = int(tiles[0])
        for have, want in zip(got[:3] + [got[3][:1 + 3 * n_tiles]], (off, srt, inv, tiles[:1 + 3 * n_tiles])):
            assert torch.equal(have, want), tokens
        assert bounds[0] == 0 and bounds[8] == n_tiles << 16 and bool((bounds[:9].diff() >= 0).all())
        if tokens <= 16:   # one wave: eight parts of equal length, every tile a block of its own (first tile << 8 | height)
            assert bounds[:9].tolist() == [(x * n_tiles) << 13 for x in range(9)]
            assert bounds[16:16 + n_tiles].tolist() == [t << 8 | 1 for t in range(n_tiles)]


def _prompt_pass_equals_small_batches(ops, g, router, b_router, t, k):
    n = lambda *s, std=1.0: (torch.randn(*s, generator=g, device="cuda") * std).bfloat16()
    E, H = router.shape
    layer = ops.MoeLayer(router, b_router, n(E, 512, H, std=0.05), n(E, 512).float(), n(E, H, 256, std=0.05), n(E, H).float(),
                         top_k=k, max_tokens=len(t))
    out = layer.forward(t).clone()                      # 512 rows per expert on average: tiles of 256
    for i in range(0, len(t), 100):
        assert torch.equal(layer.forward(t[i:i + 100].contiguous()), out[i:i + 100]), i


@pytest.mark.parametrize("rows", [1, 7, 8, 9, 250, 255, 256, 257, 263, 264, 520])
def test_last_row_tiles_of_a_prompt_pass(ops, rows):
    """Two experts, one per token: `rows` tokens take the first one."""
    g = torch.Generator(device="cuda").manual_seed(rows)
    t = torch.randn(1100, 256, generator=g, device="cuda").bfloat16()
    t[:, 0] = -1.0
    t[torch.randperm(1100, generator=g, device="cuda")[:rows], 0] = 1.0
    router = torch.zeros(2, 256, device="cuda").bfloat16()
    router[0, 0] = 1.0
    _prompt_pass_equals_small_batches(ops, g, router, torch.zeros(2, device="cuda"), t, 1)


@pytest.mark.parametrize("rows", [32, 33, 64, 65, 96, 97, 128, 129, 160, 192, 193, 224, 225, 385])
def test_row_blocks_of_a_prompt_pass(ops, rows):
    """Tiles of one to four row blocks per wave, whole and in halves (the launch has fewer tiles than workgroups)."""
    test_last_row_tiles_of_a_prompt_pass(ops, rows)


# every token on all experts: one 256-row tile from 165 rows to 248, two 160-row tiles outside; on half of them: from 213
@pytest.mark.parametrize("k,I,rows", [(4, 8640, 164), (4, 8640, 165), (4, 8640, 200), (4, 8640, 248), (4, 8640, 249),
                                      (2, 16128, 212), (2, 16128, 213), (2, 16128, 248), (2, 16128, 249)])
def test_large_blocks_of_one_and_two_row_tiles_per_expert(ops, k, I, rows):
    E, H = 4, 4096
    B = rows * E // k
    g = torch.Generator(device="cuda").manual_seed(rows)
    n = lambda *s, std=1.0: (torch.randn(*s, generator=g, device="cuda") * std).bfloat16()
    layer = ops.MoeLayer(n(E, H, std=0.02), n(E).float(), n(E, 2 * I, H, std=0.02), n(E, 2 * I).float(), n(E, H, I, std=0.02),
                         n(E, H).float(), top_k=k, max_tokens=B)
    t = n(B, H)
    out = layer.forward(t).clone()
    for i in range(0, B, 64):
        assert torch.equal(layer.forward(t[i:i + 64].contiguous()), out[i:i + 64]), i


@pytest.mark.parametrize("E,k,H,I", [(4, 4, 2048, 1024), (4, 2, 512, 256), (16, 4, 1024, 512), (4, 4, 2880, 2880)])
@pytest.mark.parametrize("rows", [33, 64, 65, 97, 129, 161, 240, 330])
def test_blocks_that_leave_cus_idle_give_the_same_in_tiles_of_any_size(ops, E, k, H, I, rows):
    """Up to 330 rows per expert where tiles of 32 to 256 rows are chosen by estimated time, against batches of 16 tokens."""
    B = rows * E // k
    g = torch.Generator(device="cuda").manual_seed(rows)
    n = lambda *s, std=1.0: (torch.randn(*s, generator=g, device="cuda") * std).bfloat16()
    layer = ops.MoeLayer(n(E, H), n(E).float(), n(E, 2 * I, H, std=0.02), n(E, 2 * I).float(), n(E, H, I, std=0.02),
                         n(E, H).float(), top_k=k, max_tokens=B)
    t = n(B, H)
    out = layer.forward(t).clone()
    for i in range(0, B, 16):
        assert torch.equal(layer.forward(t[i:i + 16].contiguous()), out[i:i + 16]), i


def _longest_tile(layer, tokens):
    """Rows of the longest row tile of the last forward call; its tile list is behind the inverse permutation."""
    ptrs = [C.c_void_p() for _ in range(6)]
    layer.L.gptoss_moe_workspace_views(layer.ws.data_ptr(), tokens, layer.E, layer.k, layer.H, layer.I, *[C.byref(p) for p in ptrs])
    at = ptrs[5].value - layer.ws.data_ptr() + (tokens * layer.k * 4 + 255) // 256 * 256
    tiles = layer.ws[at:at + 4 * (1 + 3 * (tokens * layer.k // 32 + layer.E))].view(torch.int32).tolist()
    return max(tiles[3:1 + 3 * tiles[0]:3])


# every token on all experts: 160-row tiles, or ones that are estimated to be ahead of them by 11 %
@pytest.mark.parametrize("E,H,I,rows,longest", [(4, 2880, 2880, 150, 150), (4, 2880, 2880, 165, 128), (4, 2880, 2880, 180, 128),
                                                (6, 2944, 1024, 345, 128), (2, 2816, 5056, 341, 128), (5, 2816, 4800, 70, 70)])
def test_row_tiles_where_every_token_takes_every_expert(ops, E, H, I, rows, longest):
    g = torch.Generator(device="cuda").manual_seed(rows)
    n = lambda *s, std=1.0: (torch.randn(*s, generator=g, device="cuda") * std).bfloat16()
    layer = ops.MoeLayer(n(E, H), n(E).float(), n(E, 2 * I, H, std=0.02), n(E, 2 * I).float(), n(E, H, I, std=0.02),
                         n(E, H).float(), top_k=E, max_tokens=rows)
    layer.forward(n(rows, H))
    assert _longest_tile(layer, rows) == longest


# some experts per token: 64-row tiles where they are ahead with a fifth more of them too, or with as many as there can be (four experts)
@pytest.mark.parametrize("E,k,H,I,tokens,tile", [(4, 2, 768, 2048, 845, 64), (12, 4, 512, 4672, 330, 64), (6, 2, 2624, 2688, 318, 160),
                                                 (24, 1, 2176, 768, 1332, 128)])
def test_row_tiles_where_experts_are_chosen(ops, E, k, H, I, tokens, tile):
    g = torch.Generator(device="cuda").manual_seed(tokens)
    n = lambda *s, std=1.0: (torch.randn(*s, generator=g, device="cuda") * std).bfloat16()
    layer = ops.MoeLayer(n(E, H), torch.zeros(E, device="cuda"), n(E, 2 * I, H, std=0.02), n(E, 2 * I).float(), n(E, H, I, std=0.02),
                         n(E, H).float(), top_k=k, max_tokens=tokens)
    layer.forward(n(tokens, H))
    assert _longest_tile(layer, tokens) == min(tile, int(layer.routing_views()[3].diff().max()))


@pytest.mark.parametrize("k", [1, 2, 3, 5, 7, 8])
def test_tokens_of_pairs_in_a_prompt_pass(ops, k):
    """Every token on all k experts: the token of a pair is the pair's number over k."""
    g = torch.Generator(device="cuda").manual_seed(k)
    t = torch.randn(519, 256, generator=g, device="cuda").bfloat16()
    _prompt_pass_equals_small_batches(ops, g, torch.randn(k, 256, generator=g, device="cuda").bfloat16(),
                                      torch.zeros(k, device="cuda"), t, k)
