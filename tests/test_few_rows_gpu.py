"""The few-row GEMM kernels (tiles of at most 64 rows): every row must have the bits that the streaming kernels give it
in a larger batch, at the edges of row tiles, column blocks and staged chunks of K."""
import ctypes as C

import pytest
import torch

from conftest import load_pkg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    return load_pkg("ops")


def _n(g, *shape, std=1.0):
    return (torch.randn(*shape, generator=g, device="cuda") * std).to(torch.bfloat16)


# K: one slab, one short of a chunk of eight slabs, a chunk, one more, the 20B model's; N: part of a workgroup's 128
# columns, one workgroup and a block, the 20B model's 22.5 workgroups
@pytest.mark.parametrize("K", [64, 448, 512, 576, 2880])
@pytest.mark.parametrize("N", [32, 160, 2880, 17408])   # 17408: 544 blocks in one row tile, so never a block each
def test_dense_rows_equal_those_of_a_larger_batch(ops, K, N):
    g = torch.Generator(device="cuda").manual_seed(K + N)
    a, w, bias = _n(g, 2100, K), ops.pack_weight(_n(g, N, K, std=0.05)), _n(g, N).float()
    for b in (bias, None):
        want = ops.dense_gemm(a, w, N, bias=b)     # 2100 rows: the streaming kernels, or those of 256 rows
        for rows in (1, 2, 7, 8, 9, 31, 32, 33, 63, 64, 65, 96, 130, 330):
            for first in (0, 2100 - rows):
                got = ops.dense_gemm(a[first:first + rows].contiguous(), w, N, bias=b)
                assert torch.equal(got, want[first:first + rows]), (rows, first)


def _codes(g, *shape):
    return torch.randint(0, 256, shape, generator=g, device="cuda", dtype=torch.uint8)


@pytest.mark.parametrize("H,I,E,k", [(64, 64, 4, 2), (320, 576, 8, 4), (512, 448, 4, 4), (2880, 2880, 8, 4)])
@pytest.mark.parametrize("mxfp4", [False, True])
def test_moe_rows_equal_those_of_a_larger_batch(ops, H, I, E, k, mxfp4):
    g = torch.Generator(device="cuda").manual_seed(H + I + mxfp4)
    router = (_n(g, E, H, std=H ** -0.5), _n(g, E))
    if mxfp4:
        sc = lambda *s: (127 - torch.randint(6, 10, s, generator=g, device="cuda")).to(torch.uint8)
        layer = ops.MoeLayerMxfp4(*router, _codes(g, E, 2 * I, H // 2), sc(E, 2 * I, H // 32), _n(g, E, 2 * I),
                                  _codes(g, E, H, I // 2), sc(E, H, I // 32), _n(g, E, H), top_k=k, max_tokens=512)
    else:
        layer = ops.MoeLayer(*router, _n(g, E, 2 * I, H, std=0.05), _n(g, E, 2 * I), _n(g, E, H, I, std=0.05), _n(g, E, H),
                             top_k=k, max_tokens=512)
    t = _n(g, 400, H)
    want = layer.forward(t).clone()                # 400 tokens: 200 rows per expert
    for tokens in (1, 2, 8, 9, 17, 31, 33, 60, 90):   # 9: the largest tile may have more rows than one wave stages
        got = layer.forward(t[40:40 + tokens].contiguous())
        assert torch.equal(got, want[40:40 + tokens]), tokens


def test_a_tile_list_of_one_expert_and_of_several_tiles(ops):
    """All tokens on the same experts: tiles of 32 rows with a remainder, the other experts empty."""
    g = torch.Generator(device="cuda").manual_seed(3)
    H = I = 256
    E, k = 16, 2
    b = torch.zeros(E, device="cuda")
    b[3], b[11] = 50.0, 40.0
    layer = ops.MoeLayer(_n(g, E, H, std=0.01), b, _n(g, E, 2 * I, H, std=0.05), _n(g, E, 2 * I), _n(g, E, H, I, std=0.05),
                         _n(g, E, H), top_k=k, max_tokens=512)
    t = _n(g, 512, H)
    want = layer.forward(t).clone()
    for tokens in (5, 33, 64, 70, 100):
        assert torch.equal(layer.forward(t[:tokens].contiguous()), want[:tokens]), tokens


@pytest.mark.parametrize("E,k", [(1, 1), (4, 4), (8, 3), (32, 4), (40, 8), (128, 4), (256, 8)])
@pytest.mark.parametrize("ties", [False, True])
def test_grouping_of_a_few_tokens_equals_the_sorting_kernel(ops, E, k, ties):
    """Up to 16 tokens are grouped by the router's own workgroup, beyond that by a kernel of its own."""
    g = torch.Generator(device="cuda").manual_seed(E + k)
    H = I = 64
    router = _n(g, E, H) if not ties else torch.ones(E, H, device="cuda").bfloat16()   # ties: every expert scores the same
    layer = ops.MoeLayer(router, torch.zeros(E, device="cuda"), _n(g, E, 2 * I, H), _n(g, E, 2 * I), _n(g, E, H, I),
                         _n(g, E, H), top_k=k, max_tokens=32)
    for tokens in (1, 2, 7, 15, 16, 17):
        layer.forward(_n(g, tokens, H))
        logits, w, i, off, srt, inv = layer.routing_views()
        w2, i2, off2, srt2, inv2, _ = ops.moe_route(logits, k)
        for got, want in ((w, w2), (i, i2), (off, off2), (srt, srt2), (inv, inv2)):
            assert torch.equal(got, want), tokens


# rows on both sides of where the kernel, the row tile or the number of parts changes; K: two slabs, which cannot be cut, to 128
@pytest.mark.parametrize("N,K", [(512, 128), (768, 768), (1280, 1280), (896, 4864), (2048, 8192)])
def test_products_with_their_k_cut_add_up(ops, N, K):
    """gptoss::dense_gemm_partial, which has no C entry point, by its linker name: the parts add up to the product."""
    lib = load_pkg("lib")
    f = getattr(lib.load(), "_ZN6gptoss18dense_gemm_partialEPKtS1_PfmPiiiiP12ihipStream_t")
    f.restype, f.argtypes = C.c_int, [C.c_void_p] * 3 + [C.c_size_t, C.c_void_p] + [C.c_int] * 3 + [C.c_void_p]
    g = torch.Generator(device="cuda").manual_seed(K + N)
    a, w = _n(g, 2047, K), _n(g, N, K, std=0.05)
    packed, exact = ops.pack_weight(w), a.double() @ w.double().T
    bound = K * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)     # K sums in fp32, in any order
    cut = set()
    for rows in (1, 8, 9, 32, 33, 65, 97, 257, 320, 576, 768, 1024, 1280, 1700, 2047):
        out, parts = torch.full((8 * rows * N,), float("nan"), device="cuda"), C.c_int()
        lib.check(f(a.data_ptr(), packed.data_ptr(), out.data_ptr(), out.numel(), C.byref(parts), rows, N, K,
                    torch.cuda.current_stream().cuda_stream))
        assert 1 <= parts.value <= 8
        total = out[:parts.value * rows * N].view(parts.value, rows, N).double().sum(0)
        assert bool(((total - exact[:rows]).abs() <= bound[:rows]).all()), rows
        cut.add(parts.value)
    assert cut == {1} if K == 128 else len(cut) > 1


@pytest.mark.parametrize("H,I,E,k", [(320, 2880, 8, 4), (2880, 576, 32, 4)])
def test_mxfp4_rows_of_9_to_16_tokens_equal_those_of_a_larger_batch(ops, H, I, E, k):
    g = torch.Generator(device="cuda").manual_seed(H + I)
    # exponents over the range of checkpoints, each column and each 32 inputs their own
    sc = lambda *s: (127 - torch.randint(4, 12, s, generator=g, device="cuda")).to(torch.uint8)
    layer = ops.MoeLayerMxfp4(_n(g, E, H, std=H ** -0.5), _n(g, E), _codes(g, E, 2 * I, H // 2), sc(E, 2 * I, H // 32), _n(g, E, 2 * I),
                              _codes(g, E, H, I // 2), sc(E, H, I // 32), _n(g, E, H), top_k=k, max_tokens=512)
    t = _n(g, 400, H)
    want = layer.forward(t).clone()
    for tokens in (8, 9, 10, 13, 15, 16, 17):
        assert torch.equal(layer.forward(t[50:50 + tokens].contiguous()), want[50:50 + tokens]), tokens


class _Range(C.Structure):   # gptoss::GemmBf16Range
    _fields_ = [("first", C.c_int), ("end", C.c_int), ("out", C.c_void_p), ("ld", C.c_int), ("relu_squared", C.c_int)]


# rows at the edges of the 8-, 16- and 32-row kernels; N: half blocks (3 and 320 of them), whole blocks, a workgroup of four
@pytest.mark.parametrize("N,K", [(96, 64), (96, 1088), (5120, 576), (17408, 64)])
def test_columns_that_leave_as_bf16_are_the_rounded_fp32_ones(ops, N, K):
    """gptoss::dense_gemm_mixed by its linker name: a plain and a relu-squared range beside the fp32 columns."""
    lib = load_pkg("lib")
    f = getattr(lib.load(), "_ZN6gptoss16dense_gemm_mixedEPKtS1_PfPKNS_13GemmBf16RangeEiiiiP12ihipStream_t")
    f.restype, f.argtypes = C.c_int, [C.c_void_p] * 4 + [C.c_int] * 4 + [C.c_void_p]
    g = torch.Generator(device="cuda").manual_seed(K + N)
    a, w = _n(g, 33, K), ops.pack_weight(_n(g, N, K, std=0.05))
    for rows in (1, 8, 9, 16, 17, 32, 33):
        want = ops.dense_gemm(a[:rows].contiguous(), w, N)
        out = torch.zeros(rows, N, device="cuda")
        plain, squared = (torch.zeros(rows, 40, device="cuda", dtype=torch.bfloat16) for _ in range(2))
        ranges = (_Range * 2)(_Range(0, 32, plain.data_ptr(), 40, 0), _Range(N - 32, N, squared.data_ptr(), 40, 1))
        lib.check(f(a.data_ptr(), w.data_ptr(), out.data_ptr(), ranges, 2, rows, N, K, torch.cuda.current_stream().cuda_stream))
        assert torch.equal(out[:, 32:N - 32], want[:, 32:N - 32]), rows
        assert torch.equal(plain[:, :32], want[:, :32].bfloat16()), rows
        assert torch.equal(squared[:, :32], want[:, N - 32:].relu().square().bfloat16()), rows
        assert not plain[:, 32:].any() and not squared[:, 32:].any(), rows
