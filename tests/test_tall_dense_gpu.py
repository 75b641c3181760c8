"""The 256-row kernel's dense forms by themselves, whichever kernel the estimates take at these sizes: a child process has
GPTOSS_DENSE_TALL_MIN_ROWS, which decides alone where it is set, and compares products of 2048 rows and more, which that sends to
the 256-row kernel, with the same rows in batches of a fifth, which it keeps on the others.  Same bits per row."""
import ctypes as C
import json
import os
import subprocess
import sys

import pytest

from conftest import ROOT, load_pkg

pytestmark = pytest.mark.gpu

MIN_ROWS = 2048

# Tiles of 256 rows per XCD, 32 of which are a round: 12, 25 and 3 (halves only), 74 (two rounds and halves; of the last tile's 52
# rows, 33 and 1, whose second half is 20, 1 and 0), 83 (two rounds, the rest whole); one row more than whole tiles, a column tile
# of 32 columns, K in 8 stages, not a multiple of 128
F32 = [(2500, 2880, 4096), (2049, 5120, 2880), (4096, 288, 256), (2304, 1056, 512), (2048, 2880, 4096), (2100, 16640, 256),
       (2081, 16640, 256), (2049, 16640, 256), (2369, 16672, 320)]
# columns of a plain and of a relu-squared bf16 range beside the fp32 ones, row pitches of the ranges
MIXED = [(2100, 16640, 256, 512, 8192, 8192, 16640), (2049, 2592, 320, 0, 96, 2560, 2592), (2385, 2560, 320, 64, 2560, 0, 32),
         (2304, 1056, 512, 0, 1024, 1024, 1056)]


class Range(C.Structure):   # gptoss::GemmBf16Range
    _fields_ = [("first", C.c_int), ("end", C.c_int), ("out", C.c_void_p), ("ld", C.c_int), ("relu_squared", C.c_int)]


def _f32(ops, torch, a, w, N, K):
    bias = torch.linspace(-1, 1, N, device="cuda").bfloat16().float()
    full, step = ops.dense_gemm(a, w, N, bias), len(a) // 5 + 1
    return all(torch.equal(full[r:r + step], ops.dense_gemm(a[r:r + step].contiguous(), w, N, bias)) for r in range(0, len(a), step))


def _mixed(ops, torch, a, w, N, K, p0, p1, s0, s1):
    lib = load_pkg("lib")
    f = getattr(lib.load(), "_ZN6gptoss16dense_gemm_mixedEPKtS1_PfPKNS_13GemmBf16RangeEiiiiP12ihipStream_t")
    f.restype, f.argtypes = C.c_int, [C.c_void_p] * 4 + [C.c_int] * 4 + [C.c_void_p]
    out = torch.zeros(len(a), N, device="cuda")
    plain, squared = (torch.zeros(len(a), n + 8, device="cuda", dtype=torch.bfloat16) for n in (p1 - p0, s1 - s0))
    ranges = (Range * 2)(Range(p0, p1, plain.data_ptr(), plain.shape[1], 0), Range(s0, s1, squared.data_ptr(), squared.shape[1], 1))
    lib.check(f(a.data_ptr(), w.data_ptr(), out.data_ptr(), ranges, 2, len(a), N, K, torch.cuda.current_stream().cuda_stream))
    ok, step = not plain[:, p1 - p0:].any() and not squared[:, s1 - s0:].any(), len(a) // 5 + 1
    for r in range(0, len(a), step):
        want, rows = ops.dense_gemm(a[r:r + step].contiguous(), w, N), slice(r, r + step)
        rest = [n for n in range(0, N, 32) if not (p0 <= n < p1 or s0 <= n < s1)]
        ok = (ok and torch.equal(plain[rows, :p1 - p0], want[:, p0:p1].bfloat16()) and
              torch.equal(squared[rows, :s1 - s0], want[:, s0:s1].relu().square().bfloat16()) and
              all(torch.equal(out[rows, n:n + 32], want[:, n:n + 32]) for n in rest))
    return ok


def _child():
    import torch
    ops, equal = load_pkg("ops"), {}
    for kind, cases in (("f32", F32), ("mixed", MIXED)):
        for case in cases:
            rows, N, K, *ranges = case
            g = torch.Generator(device="cuda").manual_seed(rows + N)
            a = torch.randn(rows, K, device="cuda", generator=g).bfloat16()
            w = ops.pack_weight((torch.randn(N, K, device="cuda", generator=g) * 0.05).bfloat16())
            equal[f"{kind} {case}"] = bool((_f32 if kind == "f32" else _mixed)(ops, torch, a, w, N, K, *ranges))
            print(kind, case, flush=True)
    print(json.dumps(equal))


@pytest.fixture(scope="module")
def equal(ops):
    r = subprocess.run([sys.executable, os.path.abspath(__file__)], capture_output=True, text=True, timeout=100, cwd=ROOT,
                       env=dict(os.environ, GPTOSS_DENSE_TALL_MIN_ROWS=str(MIN_ROWS)))
    assert r.returncode == 0, r.stdout + r.stderr
    return json.loads(r.stdout.splitlines()[-1])


@pytest.mark.parametrize("case", F32)
def test_rows_of_the_256_row_kernel_are_those_of_the_others(equal, case):
    assert min(case) >= 256 and case[0] >= MIN_ROWS > case[0] // 5 + 1
    assert equal[f"f32 {case}"]


@pytest.mark.parametrize("case", MIXED)
def test_its_bf16_columns_are_the_rounded_fp32_ones(equal, case):
    assert equal[f"mixed {case}"]


if __name__ == "__main__":
    _child()
