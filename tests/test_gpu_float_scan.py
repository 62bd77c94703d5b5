"""GPU: the float step over many known tokens, layer by layer (csrc/ygg_float_scan.hip through ygg_float_run_scratch and
FloatYggdrasil.run), against the float64 restatement oracle/float_oracle.py.

Bounds. In f64 a result differs from the restatement's by the order of its sums: each is of at most 528 terms, so by
about 528 eps = 1.2e-13 of the terms' size, and the recurrence's decays (at most 1) let it grow over the tokens of a case;
1e-10 as for the step kernel. In f32 528 eps = 6e-5; 2e-4 as for the step kernel, before a stream's first route that
differs.
"""
import ctypes

import numpy as np
import pytest

from oracle import float_oracle as FO
from yggdrasil_amd import _lib
from yggdrasil_amd import float_model as FM

pytestmark = pytest.mark.gpu

# n, R, R2, depth, layers, vocab, token part, state in the router, streams, tokens
CASES = [
    (64, 8, 16, 5, 3, 64, 16, True, 7, 33),      # one row per tile, as in all but the last four
    (64, 8, 16, 10, 3, 32, 16, True, 3, 16),     # more experts than rows
    (16, 5, 0, 3, 2, 27, 10, True, 5, 9),        # one block, no layer input, a token part of no whole vector
    (48, 3, 20, 4, 2, 5, 4, True, 9, 17),        # three blocks, a layer input of 20
    (96, 8, 7, 6, 3, 30, 16, False, 4, 70),      # routing on the token alone, a layer input of 7, 30 classes
    (128, 16, 32, 6, 2, 33, 16, True, 2, 130),   # 33 classes: no 16-byte rows
    (256, 33, 64, 4, 2, 40, 256, True, 5, 20),   # the widest rows: 512 router inputs, 3 rank tiles
    (64, 8, 16, 5, 1, 64, 16, True, 6, 40),      # a token layer only
    (64, 8, 16, 5, 3, 64, 16, True, 40, 420),    # 8400 rows: the route a level a step; sorted in f64, ragged tiles
    (48, 3, 20, 4, 2, 5, 4, True, 40, 440),      # sorted in f64: three blocks, a layer input of 20
    (128, 16, 32, 6, 3, 33, 16, False, 6, 720),  # sorted in f64: routing on the token alone, 33 classes
    (256, 33, 64, 4, 2, 40, 256, True, 5, 480),  # sorted in both: 512 router inputs, 3 rank tiles
]


def _layers(case, seed=11):
    n, R, R2, D, L, V, F, rs, B, T = case
    spec = FM.FloatSpec(d_state=n, block_size=16, router_depth=D, vocab=V, n_layers=L, router_token_dim=F,
                        input_rank=8, readout_rank=R, layer_input_rank=R2, router_state=rs)
    raw, ob = FM.from_params(FM.random_params(spec, seed))
    return FM.float_layers(raw), ob


def _check(r, ref, upto, tol):
    for s, t1 in enumerate(upto):
        np.testing.assert_allclose(r["logits"][s, :t1].cpu().numpy(), ref["logits"][s, :t1], rtol=tol, atol=tol)


@pytest.mark.parametrize("case", CASES, ids=[str(c) for c in CASES])
def test_scan_equals_restatement(case):
    import torch
    B, T, V = case[8], case[9], case[5]
    print(f"case {case}", flush=True)
    layers, ob = _layers(case)
    x = np.random.default_rng(1).integers(0, V, (B, T))
    first = FO.run(layers, ob, x[:, :T // 2])
    ref = FO.run(layers, ob, x[:, T // 2:], state=first["state"])
    for precision, tol in ((64, 1e-10), (32, 2e-4)):
        m = FM.FloatYggdrasil(layers, ob, precision=precision)
        st = torch.tensor(first["state"], device=m.device)
        assert _lib.lib().ygg_float_scratch(m._h, B, T - T // 2) > 0        # (else the step kernel runs)
        r = m.run(x[:, T // 2:], state=st, leaves=True, stats=True)
        torch.cuda.synchronize()
        lv = r["leaves"].cpu().numpy()
        differs = (lv != ref["leaves"]).any(-1)
        upto = [int(np.argmax(d)) if d.any() else len(d) for d in differs]
        if precision == 64:
            assert not differs.any()
            np.testing.assert_allclose(r["state"].cpu().numpy(), ref["state"], rtol=tol, atol=tol)
            np.testing.assert_allclose(r["stats"].cpu().numpy(), ref["stats"], rtol=tol, atol=0)
        else:
            assert sum(t < differs.shape[1] for t in upto) <= 1
        _check(r, ref, upto, tol)
        m.close()


@pytest.mark.parametrize("case,end,few,tol", [
    ((64, 8, 16, 5, 3, 64, 16, True, 9, 300), [300, 40, 200, 299, 0, 300, 128, 127, 300], (1, 150), 0),
    # chunks of 640 rows, sorted, and of fewer, not: their sums run in another order (bound as above)
    ((256, 33, 64, 4, 2, 40, 256, True, 9, 150), [150, 40, 100, 149, 0, 150, 128, 127, 150], (5, 130), 1e-10),
], ids=["not sorted", "sorted"])
def test_scan_in_chunks_and_bad_tokens(case, end, few, tol):
    """Scratch for a few rows only (chunks of streams and of tokens), streams that stop at a token outside [0, V) in the
    first and in a later chunk, in the last token and at once: their state is the one before it and their later rows are
    left as they were; and the same call with whole scratch gives the same values (bits, where both sort alike)."""
    import torch
    layers, ob = _layers(case)
    B, T, V = case[8], case[9], case[5]
    x = np.random.default_rng(2).integers(0, V, (B, T))
    for s, t in enumerate(end):
        if t < T:
            x[s, t] = V + s if s % 2 else -1
    m = FM.FloatYggdrasil(layers, ob, precision=64)
    L, lib = case[4], _lib.lib()
    xd = torch.tensor(x, dtype=torch.int32, device=m.device)
    got = []
    whole = lib.ygg_float_scratch(m._h, B, T)
    least = lib.ygg_float_scratch(m._h, *few)
    assert 0 < least < whole
    for size in (whole, least):
        st = m.init_state(B)
        lg = torch.full((B, T, V), 7.0, dtype=m.dtype, device=m.device)
        lv = torch.full((B, T, L), -5, dtype=torch.int32, device=m.device)
        sv = torch.zeros(L, m.stats_stride, dtype=torch.float64, device=m.device)
        ws = torch.empty(size, dtype=torch.uint8, device=m.device)
        p = [ctypes.c_void_p(t.data_ptr()) for t in (xd, st, lg, lv, sv, ws)]
        _lib.check(lib.ygg_float_run_scratch(m._h, p[0], B, T, p[1], p[2], p[3], p[4], p[5], size,
                                             ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        e = ctypes.c_uint32()
        _lib.check(lib.ygg_float_take_errors(m._h, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream),
                                             ctypes.byref(e)))
        assert e.value == 1
        got.append([t.cpu().numpy() for t in (lg, lv, st, sv)])
    for a, b in zip(*got):
        np.testing.assert_allclose(a, b, rtol=tol, atol=tol)
    lg, lv, st, _ = got[0]
    for s, t in enumerate(end):
        if t:
            ref = FO.run(layers, ob, x[s:s + 1, :t])
            np.testing.assert_allclose(lg[s, :t], ref["logits"][0], rtol=1e-10, atol=1e-10)
            np.testing.assert_array_equal(lv[s, :t], ref["leaves"][0])
            np.testing.assert_allclose(st[s], ref["state"][0], rtol=1e-10, atol=1e-10)
        else:
            assert not st[s].any()
        assert (lg[s, t:] == 7.0).all() and (lv[s, t:] == -5).all()
    assert lib.ygg_float_run_scratch(m._h, p[0], B, T, p[1], p[2], p[3], p[4], p[5], 256, None) == 5   # too little
    m.close()


def test_scratch_between_row_by_row_and_sorted():
    """A call whose rows would be sorted (8000 rows of 1024 experts in f64, past the 7400 from which a sort pays at n = 64),
    in scratch for 15 rows and more, where the sorts' arrays (135 KB) would leave none: shorter chunks, and the step
    kernel's values (bound as above)."""
    import torch
    layers, ob = _layers((64, 8, 16, 10, 3, 32, 16, True, 40, 200))
    m, lib = FM.FloatYggdrasil(layers, ob, precision=64), _lib.lib()
    B, T, V = 40, 200, 32
    x = torch.tensor(np.random.default_rng(8).integers(0, V, (B, T)), dtype=torch.int32, device=m.device)
    q = torch.cuda.current_stream().cuda_stream
    least, whole = lib.ygg_float_scratch(m._h, 1, 16), lib.ygg_float_scratch(m._h, B, T)
    got = []
    for size in (None, least, least + 60_000, least + 130_000, whole - 256, whole):
        st, lg = m.init_state(B), torch.zeros(B, T, V, dtype=m.dtype, device=m.device)
        if size is None:
            rc = lib.ygg_float_run(m._h, x.data_ptr(), B, T, st.data_ptr(), lg.data_ptr(), None, None, q)
        else:
            ws = torch.empty(size, dtype=torch.uint8, device=m.device)
            rc = lib.ygg_float_run_scratch(m._h, x.data_ptr(), B, T, st.data_ptr(), lg.data_ptr(), None, None,
                                           ws.data_ptr(), size, q)
        assert rc == 0, f"scratch of {size} bytes: {lib.ygg_last_error().decode()}"
        got.append((st.cpu().numpy(), lg.cpu().numpy()))
        for a, b in zip(got[0], got[-1]):
            np.testing.assert_allclose(b, a, rtol=1e-10, atol=1e-10)
    m.close()
