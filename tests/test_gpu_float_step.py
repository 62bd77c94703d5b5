"""GPU: the f32 step of the trained shapes (float_step in csrc/ygg_float.hip) token by token, against the float64
restatement oracle/float_oracle.py. A result's sums have at most 288 terms: 288 eps = 3.4e-5 of the terms' size, and the
decays (at most 1) let it grow over a case's tokens; 2e-4 as for the other f32 forms, before a stream's first route that
differs."""
import ctypes

import numpy as np
import pytest

from oracle import float_oracle as FO
from yggdrasil_amd import _lib
from yggdrasil_amd import float_model as FM

pytestmark = pytest.mark.gpu

# n, R, R2, depth, layers, vocab, token part, state in the router, streams
CASES = [
    (64, 8, 16, 1, 2, 64, 1, True, 3),        # one node; a token part of one
    (64, 8, 16, 5, 3, 256, 32, True, 5),      # one whole round, the widest token part, 256 classes
    (64, 8, 16, 6, 3, 33, 16, False, 5),      # two rounds, routing on the token alone
    (128, 16, 32, 5, 3, 33, 16, False, 4),    # 33 classes
    (128, 16, 32, 11, 2, 20, 7, True, 4),     # three rounds, the last of one level
    (256, 32, 64, 4, 5, 20, 32, True, 3),
    (256, 32, 64, 6, 3, 256, 5, True, 1),
    (256, 32, 64, 4, 2, 20, 33, True, 3),     # a token part of 33, past the plain build's
]
# the same shapes where the plain build does not take the call: its token part's remainder at 8, 16 and 32 lanes a node,
# the widest, no transitions (False), the maxima of a model that the plain build takes
ANY_CASES = [
    (64, 8, 16, 6, 3, 33, 33, True, 5, True),
    (64, 8, 16, 1, 2, 64, 256, False, 3, True),
    (64, 8, 16, 5, 3, 256, 16, True, 5, False),
    (128, 16, 32, 11, 2, 20, 71, True, 4, True),
    (128, 16, 32, 5, 3, 33, 16, False, 4, True),
    (128, 16, 32, 4, 5, 20, 48, True, 3, False),
    (256, 32, 64, 6, 3, 256, 256, True, 1, True),
    (256, 32, 64, 10, 2, 20, 16, True, 3, False),
    (256, 32, 64, 4, 8, 20, 32, True, 3, True),
]


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("classes,rows", [(1, 3), (27, 17), (64, 16), (65, 1), (256, 33)])
def test_nll_equals_log_softmax(classes, rows, precision):
    """ygg_float_nll against log-sum-exp in f64: the logits are exact in both, so a sum of at most 256 exponentials of
    about an ulp each and its logarithm: 1e-13 of values of at most about 200. Ends of the types, a row of one infinity
    and rows without a class (NaN)."""
    import torch
    spec = FM.FloatSpec(d_state=16, block_size=16, router_depth=2, vocab=classes, n_layers=1, router_token_dim=4,
                        input_rank=4, readout_rank=4, layer_input_rank=0)
    raw, ob = FM.from_params(FM.random_params(spec, 3))
    m = FM.FloatYggdrasil(FM.float_layers(raw), ob, precision=precision)
    rng = np.random.default_rng(classes)
    lg = (rng.normal(size=(rows, classes)) * 30).astype(np.float32 if precision == 32 else np.float64)
    lg[0, 0] = -np.inf if classes > 1 else 1.0
    if rows > 2:
        lg[1] += np.float32(3e38) if precision == 32 else 1e300
        lg[2, -1] = np.finfo(lg.dtype).min
    y = rng.integers(0, classes, rows).astype(np.int32)
    y[0] = classes - 1
    if rows > 3:
        y[3], y[4] = classes, -1
    wide = lg.astype(np.float64)
    top = wide.max(-1)
    ok = (y >= 0) & (y < classes)
    ref = np.log(np.exp(wide - top[:, None]).sum(-1)) - (wide[np.arange(rows), np.where(ok, y, 0)] - top)
    a, b = torch.tensor(lg, device=m.device), torch.tensor(y, device=m.device)
    r = torch.full((rows,), 9.0, dtype=torch.float64, device=m.device)
    _lib.check(_lib.lib().ygg_float_nll(m._h, a.data_ptr(), b.data_ptr(), rows, r.data_ptr(),
                                        torch.cuda.current_stream().cuda_stream))
    r = r.cpu().numpy()
    assert np.isnan(r[~ok]).all()
    np.testing.assert_allclose(r[ok], ref[ok], rtol=1e-13, atol=1e-13)
    m.close()


@pytest.mark.parametrize("case", CASES, ids=[str(c) for c in CASES])
def test_step_equals_restatement(case):
    import torch
    n, R, R2, D, L, V, F, rs, B = case
    print(f"case {case}", flush=True)
    spec = FM.FloatSpec(d_state=n, block_size=16, router_depth=D, vocab=V, n_layers=L, router_token_dim=F,
                        input_rank=8, readout_rank=R, layer_input_rank=R2, router_state=rs)
    raw, ob = FM.from_params(FM.random_params(spec, 5))
    layers = FM.float_layers(raw)
    T = 24
    x = np.random.default_rng(4).integers(0, V, (B, T))
    first = FO.run(layers, ob, x[:, :4])
    ref = FO.run(layers, ob, x[:, 4:], state=first["state"])
    m, lib = FM.FloatYggdrasil(layers, ob, precision=32), _lib.lib()
    assert m.kernel_name == ("ygg::float_any_kernel<%d, %d, %d>" if F > 32 else
                             "ygg::float_kernel<float, %d, %d, %d, 16>") % (n, R, R2), m.kernel_name
    end = T - 4 if B == 1 else 9                # the last stream ends at a token outside [0, V)
    if B > 1:
        x[-1, 4 + end] = V
    st = torch.tensor(first["state"], dtype=m.dtype, device=m.device)
    xd = torch.tensor(x[:, 4:], dtype=torch.int32, device=m.device).contiguous()
    lg = torch.full((B, T - 4, V), 7.0, dtype=m.dtype, device=m.device)
    lv = torch.full((B, T - 4, L), -5, dtype=torch.int32, device=m.device)
    p = [ctypes.c_void_p(t.data_ptr()) for t in (xd, st, lg, lv)]
    q = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(lib.ygg_float_run(m._h, p[0], B, T - 4, p[1], p[2], p[3], None, q))
    e = ctypes.c_uint32()
    _lib.check(lib.ygg_float_take_errors(m._h, q, ctypes.byref(e)))
    assert e.value == (1 if B > 1 else 0)
    lg, lv, st = lg.cpu().numpy(), lv.cpu().numpy(), st.cpu().numpy()
    split = 0
    for s in range(B):
        t1 = end if s == B - 1 else T - 4
        d = (lv[s, :t1] != ref["leaves"][s, :t1]).any(-1)
        upto = int(np.argmax(d)) if d.any() else t1
        split += upto < t1
        np.testing.assert_allclose(lg[s, :upto], ref["logits"][s, :upto], rtol=2e-4, atol=2e-4)
        assert (lg[s, t1:] == 7.0).all() and (lv[s, t1:] == -5).all()
        if upto == t1 == T - 4:
            np.testing.assert_allclose(st[s], ref["state"][s], rtol=2e-4, atol=2e-4)
    assert split <= 1
    m.close()


@pytest.mark.parametrize("stats", [True, False], ids=["stats", "plain"])
@pytest.mark.parametrize("case", ANY_CASES, ids=[str(c) for c in ANY_CASES])
def test_any_build_equals_restatement(case, stats):
    """The step build of a trained shape for the calls that the plain one does not take; the maxima up to 2e-4 as well,
    where no route differs."""
    import torch
    n, R, R2, D, L, V, F, rs, B, moves = case
    print(f"case {case} {stats}", flush=True)
    spec = FM.FloatSpec(d_state=n, block_size=16, router_depth=D, vocab=V, n_layers=L, router_token_dim=F,
                        input_rank=8, readout_rank=R, layer_input_rank=R2, router_state=rs)
    p = {k: v for k, v in FM.random_params(spec, 6).items() if moves or k.rsplit("/")[-1] not in ("rotation", "decay")}
    raw, ob = FM.from_params(p)
    layers = FM.float_layers(raw)
    T = 16
    x = np.random.default_rng(5).integers(0, V, (B, T + 4))
    first = FO.run(layers, ob, x[:, :4])
    ref = FO.run(layers, ob, x[:, 4:], state=first["state"])
    m, lib = FM.FloatYggdrasil(layers, ob, precision=32), _lib.lib()
    plain = moves and F <= 32
    assert m.kernel_name == ("ygg::float_kernel<float, %d, %d, %d, 16>" if plain else
                             "ygg::float_any_kernel<%d, %d, %d>") % (n, R, R2), m.kernel_name
    st = torch.tensor(first["state"], dtype=m.dtype, device=m.device)
    xd = torch.tensor(x[:, 4:], dtype=torch.int32, device=m.device).contiguous()
    lg = torch.empty(B, T, V, dtype=m.dtype, device=m.device)
    lv = torch.empty(B, T, L, dtype=torch.int32, device=m.device)
    sv = torch.zeros(L, m.stats_stride, dtype=torch.float64, device=m.device)
    _lib.check(lib.ygg_float_run(m._h, xd.data_ptr(), B, T, st.data_ptr(), lg.data_ptr(), lv.data_ptr(),
                                 sv.data_ptr() if stats else None, torch.cuda.current_stream().cuda_stream))
    lg, lv, st, sv = (t.cpu().numpy() for t in (lg, lv, st, sv))
    split = 0
    for s in range(B):
        d = (lv[s] != ref["leaves"][s]).any(-1)
        upto = int(np.argmax(d)) if d.any() else T
        split += upto < T
        np.testing.assert_allclose(lg[s, :upto], ref["logits"][s, :upto], rtol=2e-4, atol=2e-4)
        if upto == T:
            np.testing.assert_allclose(st[s], ref["state"][s], rtol=2e-4, atol=2e-4)
    assert split <= 1
    if stats and not split:
        np.testing.assert_allclose(sv, ref["stats"], rtol=2e-4, atol=0)
    assert stats or not sv.any()
    m.close()


@pytest.mark.parametrize("precision,tol", [(32, 2e-4), (64, 1e-10)])
@pytest.mark.parametrize("n,b", [(16, 1), (32, 2), (48, 4), (64, 8), (96, 16), (48, 3)])
def test_general_kernel_blocks(n, b, precision, tol):
    """The general kernel's transition blocks of each size, in the layouts that f32 and f64 store them in (bounds as
    above, 1e-10 in f64)."""
    spec = FM.FloatSpec(d_state=n, block_size=b, router_depth=3, vocab=20, n_layers=2, router_token_dim=8, input_rank=8,
                        readout_rank=5, layer_input_rank=7)
    raw, ob = FM.from_params(FM.random_params(spec, 8))
    layers = FM.float_layers(raw)
    x = np.random.default_rng(6).integers(0, 20, (4, 3))
    ref = FO.run(layers, ob, x)
    m = FM.FloatYggdrasil(layers, ob, precision=precision)
    r = m.run(x, leaves=True)
    lv = r["leaves"].cpu().numpy()
    np.testing.assert_array_equal(lv, ref["leaves"])
    np.testing.assert_allclose(r["logits"].cpu().numpy(), ref["logits"], rtol=tol, atol=tol)
    np.testing.assert_allclose(r["state"].cpu().numpy(), ref["state"], rtol=tol, atol=tol)
    m.close()
