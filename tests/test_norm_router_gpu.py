"""The MoE block that runs the residual add and RMSNorm in front of it by itself, as the engine calls it: every result
must have the bits of the norm, the router, the grouping and the block called one after the other."""
import ctypes as C

import pytest
import torch

from conftest import load_pkg

pytestmark = pytest.mark.gpu


class _PreNorm(C.Structure):   # MoePreNorm of gemm.hpp
    _fields_ = [("x", C.c_void_p), ("residual", C.c_void_p), ("weight", C.c_void_p)]


def _forward_norm(layer, x, residual, weight, out, next_weight=None, next_t=None):
    """gptoss::moe_forward_norm, which has no C entry point, by its linker name; -> its t, bf16 [B, H].  With next_weight
    the norm of the updated rows goes to next_t."""
    f = getattr(layer.L, "_ZN6gptoss16moe_forward_normEPK18gptoss_moe_weightsPKviPfPvmP12ihipStream_tiPKfPtPKNS_10MoePreNormE")
    f.restype = C.c_int
    f.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_void_p, C.c_void_p, C.c_size_t, C.c_void_p, C.c_int, C.c_void_p,
                  C.c_void_p, C.c_void_p]
    B, H = x.shape
    assert B <= layer.max_tokens and all(v.is_contiguous() for v in (x, weight, out))
    assert residual is None or (residual.shape == x.shape and residual.is_contiguous())
    t = torch.empty(B, H, dtype=torch.bfloat16, device="cuda")
    pre = _PreNorm(x.data_ptr(), residual.data_ptr() if residual is not None else None, weight.data_ptr())
    behind = (None, None) if next_weight is None else (next_weight.data_ptr(), next_t.data_ptr())
    load_pkg("lib").check(f(C.byref(layer.desc), t.data_ptr(), B, out.data_ptr(), layer.ws.data_ptr(), layer.ws_bytes,
                            torch.cuda.current_stream().cuda_stream, 0, *behind, C.byref(pre)))
    layer._last_B = B
    return t


# H: a part of a thread's first chunk, three chunks short of the end, four whole chunks; E: one column block, two, four, eight,
# sixteen of the kernel's instances
@pytest.mark.parametrize("H", [64, 2880, 4096])
@pytest.mark.parametrize("E", [4, 32, 33, 64, 128, 129])
@pytest.mark.parametrize("with_residual", [False, True])
def test_a_block_with_its_norm_equals_its_parts(ops, H, E, with_residual):
    check_block_with_its_norm(ops, H, E, with_residual)


# the router's two sets of k-steps per wave: up to 32 experts 1536 inputs each, up to 64 1024, up to 128 512 (beyond, one set of
# 512); just below a set's end, at it and behind it, where the second one begins or the first is filled again
@pytest.mark.parametrize("E,H", [(E, end + d) for E, ends in ((16, (1536, 3072)), (32, (1536, 3072)), (33, (1024, 2048)), (64, (1024, 2048)),
                                                              (65, (512, 1024, 1536)), (128, (512, 1024, 1536)), (129, (512, 1024)))
                                 for end in ends for d in (-64, 0, 64)])
def test_a_block_with_its_norm_at_the_ends_of_the_routers_sets(ops, E, H):
    check_block_with_its_norm(ops, H, E, True)


def check_block_with_its_norm(ops, H, E, with_residual):
    g = torch.Generator(device="cuda").manual_seed(H + E)
    rnd = lambda *s, std=1.0: torch.randn(*s, generator=g, device="cuda") * std
    n = lambda *s, **k: rnd(*s, **k).bfloat16()
    I = 64
    layer = ops.MoeLayer(n(E, H, std=H ** -0.5), n(E), n(E, 2 * I, H, std=0.05), n(E, 2 * I), n(E, H, I, std=0.05), n(E, H),
                         top_k=4, max_tokens=601)
    weight = 1 + rnd(H, std=0.1)
    # 1, 2, 3, 4 rows: one workgroup groups them; 5, 16, 17: several, and a launch that sorts; 301: a last one of one row.  33 and
    # more experts of H = 2880 and 4096 are shared out among workgroups, behind a norm of its own, up to 512 rows; from 513
    # on, and at H = 64 always, the norm runs in the router's kernel for them too, with four rows per workgroup
    for B in (1, 2, 3, 4, 5, 16, 17, 301, 513, 601):
        x, residual = rnd(B, H) * 3, rnd(B, H) if with_residual else None
        x_want, out = x.clone(), rnd(B, H)
        out_want = out.clone()
        t = _forward_norm(layer, x, residual, weight, out)
        got = [x, t, out] + layer.routing_views()
        t_want = ops.rmsnorm(x_want, weight, residual)
        logits = ops.router_gemm(t_want, layer.w_router, layer.b_router)
        w, ids, offsets, order, place, _ = ops.moe_route(logits, 4)
        layer.forward(t_want, out=out_want, accumulate=True)
        want = [x_want, t_want, out_want, logits, w, ids, offsets, order, place]
        for name, a, b in zip("x t out logits weights ids offsets order place".split(), got, want):
            assert torch.equal(a, b), (B, name)


# k: places for four experts and for eight; H: every number of chunks per thread that the fused kernel has
@pytest.mark.parametrize("k", [1, 4, 5, 8])
@pytest.mark.parametrize("H", [64, 1024, 2048, 2880, 4096])
def test_a_block_with_the_norm_behind_it_equals_its_parts(ops, k, H):
    g = torch.Generator(device="cuda").manual_seed(H + k)
    rnd = lambda *s, std=1.0: torch.randn(*s, generator=g, device="cuda") * std
    n = lambda *s, **kw: rnd(*s, **kw).bfloat16()
    E, I, B = 16, 64, 23
    layer = ops.MoeLayer(n(E, H, std=H ** -0.5), n(E), n(E, 2 * I, H, std=0.05), n(E, 2 * I), n(E, H, I, std=0.05), n(E, H),
                         top_k=k, max_tokens=B)
    weight, next_weight = 1 + rnd(H, std=0.1), 1 + rnd(H, std=0.1)
    x, residual = rnd(B, H) * 3, rnd(B, H)
    want = x.clone()
    got_t = torch.empty(B, H, dtype=torch.bfloat16, device="cuda")
    _forward_norm(layer, x, residual, weight, x, next_weight, got_t)       # accumulates into x, as the engine has it
    layer.forward(ops.rmsnorm(want, weight, residual), out=want, accumulate=True)
    assert torch.equal(x, want)
    assert torch.equal(got_t, ops.rmsnorm(want, next_weight))
