"""The delta rules and the state-space recurrence over the rows of a step, in the form that a step takes (stretches of a prompt:
the state-space recurrence in chunks on the matrix cores) and token by token, against the recurrence in 64 bits:
gptoss::run_scan_chunks and gptoss::run_scan by their linker names, at the edges of chunks, key and column blocks."""
import ctypes as C

import numpy as np
import pytest
import torch

from conftest import load_pkg

pytestmark = pytest.mark.gpu

DELTA, CHANNEL_DELTA, STATE_SPACE = 0, 1, 2


def _struct(name, *fields):
    return type(name, (C.Structure,), {"_fields_": [(f, {"i": C.c_int, "f": C.c_float, "p": C.c_void_p}.get(t, t))
                                                    for t, names in fields for f in names.split()]})


Rotary = _struct("Rotary", ("p", "table"), ("i", "dims interleaved"))
ShortConv = _struct("ShortConv", ("i", "col channels taps"), ("p", "weight bias"), ("i", "n_unit unit_dim"), ("f", "unit_scale"))
Scan = _struct("Scan", ("i", "kind heads key_heads K V"), ("p", "conv"), ("i", "ld_conv q_col k_col v_col"), ("p", "inp"),
               ("i", "ld_in beta_col decay_col"), ("p", "channel_decay"), ("i", "ld_decay"),
               ("p", "a_log dt_bias d_skip head_decay decay_powers"), ("f", "value_scale"), (Rotary, "rot"),
               ("p", "state out"), ("i", "ld_out"), (ShortConv, "conv_desc"), ("p", "conv_state"), ("i", "vec"))
StepRows = _struct("StepRows", ("i", "n n_seg max_len"), ("p", "tokens slots lens offset segs sample singles"),
                   ("i", "n_singles longest"), ("p", "tiles0 tiles1 tiles2"))


def _takes_chunks(lib, p, r):
    f = lib["_ZN6gptoss17scan_chunks_applyERKNS_4ScanERKNS_8StepRowsE"]
    f.restype, f.argtypes = C.c_bool, [C.c_void_p, C.c_void_p]
    return f(C.addressof(p), C.addressof(r))


def _softplus(x):
    return np.maximum(x, 0) + np.log1p(np.exp(-np.abs(x)))


def _exact(kind, q, k, v, b, a, rate, bias, skip, S):
    """-> outputs [T, H, V], state [H, V, K], from state S, in float64."""
    T, H, V = v.shape
    out, dt = np.zeros((T, H, V)), _softplus(a + bias)
    decay = np.exp(-rate.reshape(H, 1) * dt.reshape(T, H, -1))   # one, or one per key channel
    for t in range(T):
        S = S * decay[t][:, None, :]
        if kind != STATE_SPACE:
            u = (v[t] - np.einsum("hvk,hk->hv", S, k[t])) / (1 + np.exp(-b[t]))[:, None]
        else:
            u = dt[t][:, None] * v[t]
        S = S + u[:, :, None] * k[t][:, None, :]
        out[t] = np.einsum("hvk,hk->hv", S, q[t]) + (skip[:, None] * v[t] if kind == STATE_SPACE else 0)
    return out, S


def _both_forms(kind, heads, key_heads, K, V, conv, inp, a, a_log, bias, skip, state, segs, short_conv=None,
                conv_state=None):
    """-> outputs [T, heads, V], states and convolution states in the form that a step takes, then token by token, in float64."""
    n, longest = len(conv), int(segs[:, 1].max())
    lib, keep = load_pkg("lib").load(), []

    def dev(x):
        keep.append(torch.from_numpy(np.ascontiguousarray(x)).cuda())
        return keep[-1].data_ptr()

    nk = key_heads * K
    got = []
    chunks, tokens = (getattr(lib, name) for name in ("_ZN6gptoss15run_scan_chunksERKNS_4ScanERKNS_8StepRowsEP12ihipStream_t",
                                                      "_ZN6gptoss8run_scanERKNS_4ScanERKNS_8StepRowsEP12ihipStream_t"))
    for f in (chunks, tokens):
        st, out = torch.from_numpy(state).cuda(), torch.full((n, heads * V), np.nan, device="cuda")
        taken = torch.from_numpy(conv_state if conv_state is not None else np.zeros(1, np.float32)).cuda()
        p = Scan(kind=kind, heads=heads, key_heads=key_heads, K=K, V=V, conv=dev(conv), ld_conv=conv.shape[1], q_col=0, k_col=nk,
                 v_col=2 * nk, inp=dev(inp), ld_in=inp.shape[1], beta_col=0, decay_col=heads,
                 channel_decay=dev(a) if kind == CHANNEL_DELTA else None, ld_decay=heads * K, a_log=dev(a_log), dt_bias=dev(bias),
                 d_skip=dev(skip), value_scale=1.0, state=st.data_ptr(), out=out.data_ptr(), ld_out=heads * V,
                 conv_desc=short_conv or ShortConv(taps=1), conv_state=taken.data_ptr())
        singles = segs[segs[:, 1] == 1]
        r = StepRows(n=n, n_seg=len(segs), segs=dev(segs), singles=dev(singles) if len(singles) else None, n_singles=len(singles),
                     longest=longest)
        if f is chunks and not _takes_chunks(lib, p, r):
            f = tokens
        f.restype, f.argtypes = C.c_int, [C.c_void_p, C.c_void_p, C.c_void_p]
        torch.cuda.synchronize()
        assert f(C.addressof(p), C.addressof(r), None) == 0
        torch.cuda.synchronize()
        got.append([x.cpu().numpy().astype(np.float64) for x in (out.view(n, heads, V), st, taken)])

    return got


@pytest.mark.parametrize("strong", [False, True])
@pytest.mark.parametrize("kind", [DELTA, CHANNEL_DELTA, STATE_SPACE])
@pytest.mark.parametrize("heads,key_heads,K,V,lengths", [
    (2, 1, 4, 5 * 4, (48, 1, 49)),          # one key block of which an eighth is there; a token beside the stretches
    (4, 2, 36, 68, (64, 65, 31)),           # two column blocks, the second of four columns
    (2, 2, 128, 64, (95, 96, 97, 32, 33)),
    (1, 1, 132, 128, (50,)),
    (2, 1, 160, 20, (63, 17, 48)),
    (2, 1, 256, 16, (129, 15, 16, 17)),     # the largest keys
    (6, 3, 64, 64, (70,) + 100 * (1,)),
])
def test_chunks_equal_the_recurrence(kind, strong, heads, key_heads, K, V, lengths):
    g = np.random.default_rng(K + V + kind)
    n, slots, KP = sum(lengths), len(lengths), (K + 31) // 32 * 32
    unit = lambda x: x / np.sqrt((x * x).sum(-1, keepdims=True))
    q, k = unit(g.standard_normal((n, key_heads, K))) / np.sqrt(K), unit(g.standard_normal((n, key_heads, K)))
    v = g.standard_normal((n, heads, V))
    channels = (heads, K) if kind == CHANNEL_DELTA else (heads,)
    b, a = g.standard_normal((n, heads)), g.standard_normal((n, *channels))
    a_log, bias, skip = g.uniform(-5, -.5, heads) + 4.5 * strong, g.standard_normal(channels), g.standard_normal(heads)
    state = np.zeros((slots, heads, V, KP))
    state[..., :K] = g.standard_normal((slots, heads, V, K)) * 0.1
    f32 = lambda x: np.ascontiguousarray(x, np.float32)
    q, k, v, b, a, a_log, bias, skip, state = map(f32, (q, k, v, b, a, a_log, bias, skip, state))
    conv = np.concatenate([q.reshape(n, -1), k.reshape(n, -1), v.reshape(n, -1)], axis=1)
    inp = np.concatenate([b, a.reshape(n, -1)], axis=1)
    order = g.permutation(slots)               # slots in another order than the stretches; the first starts from nothing
    at = np.concatenate([[0], np.cumsum(lengths)])[:-1]
    segs = np.array([(r, m, s, 0 if i == 0 else 7) for i, (r, m, s) in enumerate(zip(at, lengths, order))], np.int32)

    got = _both_forms(kind, heads, key_heads, K, V, conv, inp, a, a_log, bias, skip, state, segs)

    d = lambda x: x.astype(np.float64)
    rep = lambda x: np.repeat(d(x), heads // key_heads, axis=1)
    want, state_want = np.zeros((n, heads, V)), d(state)
    for r0, m, s, pos0 in segs:
        rows = slice(r0, r0 + m)
        S0 = d(state[s, ..., :K]) if pos0 else np.zeros((heads, V, K))
        want[rows], state_want[s, ..., :K] = _exact(kind, rep(q)[rows], rep(k)[rows], d(v)[rows], d(b)[rows], d(a)[rows],
                                                    np.exp(d(a_log)), d(bias), d(skip), S0)
    state_want[order[0], ..., K:] = 0
    # A sum of K products and of a chunk's tokens, and a decay per token, in fp32: a few hundred roundings of 6e-8 that add up
    # like their root, 2e-6 of the largest value; the two forms are alike in that.
    for out, st, _ in got:
        assert np.isfinite(out).all()
        assert np.abs(out - want).max() <= 4e-6 * np.abs(want).max()
        assert np.abs(st - state_want).max() <= 4e-6 * np.abs(state_want).max()
    rms = [np.sqrt(((out - want) ** 2).mean()) for out, _, _ in got]
    assert rms[0] <= 1.5 * rms[1] + 1e-8


@pytest.mark.parametrize("what", ["value", "decay"])
@pytest.mark.parametrize("kind", [DELTA, CHANNEL_DELTA, STATE_SPACE])
def test_an_infinity_reaches_no_earlier_token(kind, what):
    """A value that is infinite spoils its column from its token on and nothing in front of it; a decay input that is (of a
    channel, where there is one for each) only empties the state."""
    g = np.random.default_rng(7 + kind)
    n, H, K, V, bad = 70, 2, 64, 64, 37
    unit = lambda x: x / np.sqrt((x * x).sum(-1, keepdims=True))
    f32 = lambda x: np.ascontiguousarray(x, np.float32)
    q, k, v = unit(g.standard_normal((n, H, K))), unit(g.standard_normal((n, H, K))), g.standard_normal((n, H, V))
    b, a = g.standard_normal((n, H)), g.standard_normal((n, H, K) if kind == CHANNEL_DELTA else (n, H))
    bias, state = g.standard_normal(a.shape[1:]), np.zeros((1, H, V, K), np.float32)
    if what == "value":
        v[bad, 1, 5] = np.inf
    elif kind == STATE_SPACE:   # (the input is its step size too, of what it writes)
        a[bad, 1] = 1e30
    else:
        a[bad, 1] = np.inf
    conv = f32(np.concatenate([q.reshape(n, -1), k.reshape(n, -1), v.reshape(n, -1)], axis=1))
    inp = f32(np.concatenate([b, a.reshape(n, -1)], axis=1))
    (got, _, _), (want, _, _) = _both_forms(kind, H, H, K, V, conv, inp, f32(a), f32(g.uniform(-3, -1, H)), f32(bias),
                                      f32(g.standard_normal(H)), state, np.array([(0, n, 0, 0)], np.int32))
    fine = np.ones((n, H, V), bool)
    if what == "value":
        fine[bad:, 1, 5] = False
    elif kind == STATE_SPACE:
        fine[bad:, 1] = False   # 1e30 times as large as the others
    assert np.isfinite(want[fine]).all() and np.isfinite(got[fine]).all()
    assert np.abs(got - want)[fine].max() <= 8e-6 * np.abs(want[fine]).max()   # either form's 4e-6


def _drift(g, *shape):
    return g.standard_normal((1, *shape[1:])) + 0.1 * np.cumsum(g.standard_normal(shape), axis=0)


def _taps_and_silu(g, *shape):
    taps, x = g.standard_normal((4, *shape[1:])) / 2, g.standard_normal((shape[0] + 3, *shape[1:]))
    y = sum(taps[i] * x[i:i + shape[0]] for i in range(4))
    return y / (1 + np.exp(-y))


KEYS = {"random": lambda g, *shape: g.standard_normal(shape), "as a model makes them": _taps_and_silu, "drifting": _drift,
        "with a common part": lambda g, *shape: g.standard_normal((1, *shape[1:])) + 0.3 * g.standard_normal(shape)}


@pytest.mark.parametrize("strong", [False, True])
@pytest.mark.parametrize("keys", KEYS)
@pytest.mark.parametrize("kind", [DELTA, CHANNEL_DELTA, STATE_SPACE])
def test_the_form_of_a_prompt_is_as_exact_as_token_by_token(kind, keys, strong):
    """Errors of the outputs against 64 bits, where keys are random, as the layers make them, or agree (then a delta rule takes off
    most of what the state holds): three sizes together, within a tenth, by which two correct orders of the sums differ."""
    ratios = []
    for heads, K, V in ((4, 128, 64), (4, 64, 64), (2, 256 if kind != CHANNEL_DELTA else 160, 32)):
        g, n = np.random.default_rng(K), 320
        unit = lambda x: x / np.sqrt((x * x).sum(-1, keepdims=True)) * (np.sqrt(K) if kind == STATE_SPACE else 1)
        f32 = lambda x: np.ascontiguousarray(x, np.float32)
        k = unit(KEYS[keys](g, n, heads, K))   # a delta rule's are unit vectors; the state space's channels are of size 1
        q = unit(k + 0.3 * unit(g.standard_normal(k.shape)) if keys != "random" else g.standard_normal(k.shape)) / np.sqrt(K)
        channels = (heads, K) if kind == CHANNEL_DELTA else (heads,)
        v, b, a = g.standard_normal((n, heads, V)), g.standard_normal((n, heads)), g.standard_normal((n, *channels))
        q, k, v, b, a, rate, bias, skip = map(f32, (q, k, v, b, a, g.uniform(-5, -.5, heads) + 4.5 * strong,
                                                    g.standard_normal(channels), g.standard_normal(heads)))
        state = np.zeros((1, heads, V, (K + 31) // 32 * 32), np.float32)
        conv = np.concatenate([q.reshape(n, -1), k.reshape(n, -1), v.reshape(n, -1)], axis=1)
        got = _both_forms(kind, heads, heads, K, V, conv, np.concatenate([b, a.reshape(n, -1)], axis=1), a, rate, bias, skip, state,
                          np.array([(0, n, 0, 0)], np.int32))
        d = lambda x: x.astype(np.float64)
        want, _ = _exact(kind, d(q), d(k), d(v), d(b), d(a), np.exp(d(rate)), d(bias), d(skip), np.zeros((heads, V, K)))
        ratios.append(np.divide(*(np.sqrt(((out - want) ** 2).mean()) for out, _, _ in got)))
    assert np.mean(ratios) <= 1.1, ratios


@pytest.mark.parametrize("kind", [DELTA, CHANNEL_DELTA, STATE_SPACE])
@pytest.mark.parametrize("lengths", [(48, 1, 47), (1, 300, 1), (2, 64, 1, 49, 31), (70,) + 100 * (1,), (48, 50)])
def test_short_stretches_beside_a_prompt_are_as_alone(kind, lengths):
    """A stretch's form depends on its own length only: those of fewer than 48 rows have the bits that they have token by token,
    whatever else is in the step.  The convolution's state of every stretch is brought up to date once: the last three inputs,
    those in front of the stretch from the state as it was, or zero where the sequence begins."""
    g = np.random.default_rng(sum(lengths) + kind)
    n, slots, H, K, V, taps, channels = sum(lengths), len(lengths), 2, 64, 68, 4, 300
    f32 = lambda x: np.ascontiguousarray(x, np.float32)
    unit = lambda x: x / np.sqrt((x * x).sum(-1, keepdims=True))
    a = g.standard_normal((n, H, K) if kind == CHANNEL_DELTA else (n, H))
    conv = f32(np.concatenate([unit(g.standard_normal((n, 2 * H, K))).reshape(n, -1), g.standard_normal((n, H * V))], axis=1))
    before = np.concatenate([g.standard_normal((n, H)), a.reshape(n, -1)], axis=1)
    x = f32(g.standard_normal((n, channels)))
    at = np.concatenate([[0], np.cumsum(lengths)])[:-1]
    segs = np.array([(r, m, s, 0 if i == 1 else 2 + i) for i, (r, m, s) in enumerate(zip(at, lengths, g.permutation(slots)))], np.int32)
    state, taken = f32(g.standard_normal((slots, H, V, K))), f32(g.standard_normal((slots, taps - 1, channels)))
    got = _both_forms(kind, H, H, K, V, conv, np.concatenate([f32(before), x], axis=1), f32(a), f32(g.uniform(-3, -1, H)),
                      f32(g.standard_normal(a.shape[1:])), f32(g.standard_normal(H)), state, segs,
                      ShortConv(col=before.shape[1], channels=channels, taps=taps), taken)
    (out, st, left), (out_alone, st_alone, left_alone) = got
    for r, m, s, pos0 in segs:
        if m < 48:
            assert np.array_equal(out[r:r + m], out_alone[r:r + m]) and np.array_equal(st[s], st_alone[s])
        older = taken[s] if pos0 else np.zeros_like(taken[s])
        assert np.array_equal(left[s], np.concatenate([older, x[r:r + m]])[-(taps - 1):])
    assert np.array_equal(left, left_alone)
    assert np.abs(out - out_alone).max() <= 8e-6 * np.abs(out_alone).max()   # either form's 4e-6
