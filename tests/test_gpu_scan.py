"""GPU: the int8 step over many known tokens, layer by layer (csrc/ygg_scan.hip through ygg_run_scratch and
ygg_score_scratch, Yggdrasil.run and score), against the oracle: leaves, logits and states bit for bit, the score to 1e-12
as for the step kernels."""
import ctypes

import numpy as np
import pytest

from oracle.oracle import Oracle
from yggdrasil_amd import synth

pytestmark = pytest.mark.gpu

K = synth.ModelSpec
# a model and its streams and tokens: every width, layer count, storage and scale mode, ragged tiles, tokens about the
# scan's 8 and 16 ahead; each row by row and with the rows sorted by expert
CASES = [
    (K(64, 16, 5, 256, 2, 8, 16), 3, 16),
    (K(64, 16, 5, 27, 5, 8, 16), 5, 17),
    (K(64, 16, 4, 5, 3, 8, 16, group=True), 1, 49),
    (K(96, 16, 6, 5, 3, 8, 16), 7, 40),
    (K(96, 16, 13, 5, 3, 8, 16), 2, 9),
    (K(128, 16, 7, 256, 4, 8, 16, router="gauss"), 9, 64),
    (K(128, 16, 14, 64, 2, 8, 16, router="gauss"), 3, 31),
    (K(128, 16, 6, 33, 5, 16, 32, group=True), 6, 33),
    (K(128, 16, 6, 256, 5, 16, 32, input_rank=32), 11, 50),
    (K(128, 16, 5, 27, 2, 16, 32, input_rank=64, group=True), 4, 7),
    (K(256, 16, 6, 256, 5, 32, 64), 5, 130),
    (K(256, 16, 4, 5, 3, 32, 64, group=True), 2, 2),
    (K(256, 16, 3, 27, 4, 32, 64, input_rank=64), 3, 35),
    (K(128, 16, 9, 256, 3, 8, 16, router="skew", hot_levels=7), 40, 200),
]


def _bits(logits, y):
    lg = logits.astype(np.float64)
    mx = lg.max(-1, keepdims=True)
    lse = np.log(np.exp(lg - mx).sum(-1)) + mx[..., 0]
    return (lse - np.take_along_axis(lg, y[..., None], -1)[..., 0]).sum(-1) / np.log(2)


@pytest.mark.parametrize("mode", ["1", "sort"])
@pytest.mark.parametrize("case", CASES, ids=[f"{c[0].d_state}-{i}" for i, c in enumerate(CASES)])
def test_scan_equals_oracle(case, mode, tmp_path, monkeypatch):
    import torch
    from yggdrasil_amd import _lib
    from yggdrasil_amd.inference import Yggdrasil
    spec, B, T = case
    print(f"case {case} {mode}", flush=True)
    monkeypatch.setenv("YGG_SCAN", mode)
    p = tmp_path / "m.bin"
    synth.write_model(spec, 5, p)
    m, o = Yggdrasil.load(p), Oracle(str(p))
    x = np.random.default_rng(B * T).integers(0, spec.vocab, (B, T + 3)).astype(np.int32)
    first = o.run(x[:, :3], states=True)
    st = np.ascontiguousarray(first["states"][:, -1])
    ref = o.run(x[:, 3:], state=st, states=True)
    assert _lib.lib().ygg_scratch(m._h, B, T, 0) > 0
    r = m.run(x[:, 3:], state=torch.as_tensor(st, device=m.device), leaves=True)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(r["leaves"].cpu().numpy(), ref["leaves"])
    np.testing.assert_array_equal(r["logits"].cpu().numpy(), ref["logits"])
    np.testing.assert_array_equal(r["state"].cpu().numpy(), ref["states"][:, -1])
    bits = m.score(x[:, 3:], state=torch.as_tensor(st, device=m.device))
    np.testing.assert_allclose(bits, _bits(ref["logits"][:, :-1], x[:, 4:].astype(np.int64)), rtol=1e-12)
    # the state alone
    s2 = m.run(x[:, 3:], state=torch.as_tensor(st, device=m.device), logits=False)["state"]
    np.testing.assert_array_equal(s2.cpu().numpy(), ref["states"][:, -1])
    m.close()


@pytest.mark.parametrize("spec,mode", [(K(128, 16, 5, 64, 3, 8, 16), "sort"), (K(64, 16, 13, 27, 2, 8, 16), "1")])
def test_scan_in_chunks_and_bad_tokens(spec, mode, tmp_path, monkeypatch):
    """Scratch for a few rows only (chunks of streams and of tokens), streams that stop at a token outside [0, V) and a
    target outside it: the streams' states, rows and NLL as the token-by-token calls give them, rows past a stream's
    end left as they were, and the same bits with whole scratch."""
    import torch
    from yggdrasil_amd import _lib
    from yggdrasil_amd.inference import Yggdrasil
    monkeypatch.setenv("YGG_SCAN", mode)
    p = tmp_path / "m.bin"
    synth.write_model(spec, 6, p)
    m, lib = Yggdrasil.load(p), _lib.lib()
    B, T, V, L = 9, 300, spec.vocab, spec.n_layers
    rng = np.random.default_rng(3)
    x, y = rng.integers(0, V, (B, T)), rng.integers(0, V, (B, T))
    end = [T, 40, 200, T - 1, 0, T, 128, 127, T]
    for s, t in enumerate(end):
        if t < T:
            x[s, t] = V + s if s % 2 else -1
    y[2, 7] = V
    y[5, 299] = -1
    dev = lambda a: torch.tensor(a, dtype=torch.int32, device=m.device)  # noqa: E731
    xd, yd = dev(x), dev(y)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    q = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    err = ctypes.c_uint32()
    got = []
    for size in (None, lib.ygg_scratch(m._h, B, T, 1), lib.ygg_scratch(m._h, 1, 150, 1)):
        st, st2 = m.init_state(B), m.init_state(B)
        lg = torch.full((B, T, V), 7.0, device=m.device)
        lv = torch.full((B, T, L), -5, dtype=torch.int32, device=m.device)
        nll = torch.ones(B, dtype=torch.float64, device=m.device)
        if size is None:
            _lib.check(lib.ygg_run(m._h, ptr(xd), B, T, ptr(st), ptr(lg), ptr(lv), None, None, q))
            _lib.check(lib.ygg_score(m._h, ptr(xd), ptr(yd), B, T, ptr(st2), ptr(nll), q))
        else:
            ws = torch.empty(size, dtype=torch.uint8, device=m.device)
            _lib.check(lib.ygg_run_scratch(m._h, ptr(xd), B, T, ptr(st), ptr(lg), ptr(lv), ptr(ws), size, q))
            _lib.check(lib.ygg_score_scratch(m._h, ptr(xd), ptr(yd), B, T, ptr(st2), ptr(nll), ptr(ws), size, q))
        _lib.check(lib.ygg_take_errors(m._h, q, ctypes.byref(err)))
        assert err.value == 3
        got.append([t.cpu().numpy() for t in (lg, lv, st, st2, nll)])
    for other in got[1:]:
        for a, b in zip(got[0], other):
            np.testing.assert_array_equal(a, b)
    lg, lv = got[0][:2]
    for s, t in enumerate(end):
        assert (lg[s, t:] == 7.0).all() and (lv[s, t:] == -5).all()
    assert lib.ygg_run_scratch(m._h, ptr(xd), B, T, ptr(st), ptr(lg := torch.empty(1, device=m.device)), None, ptr(ws),
                               256, q) == 5                                        # too little scratch
    m.close()


@pytest.mark.parametrize("score", [0, 1])
def test_scratch_between_row_by_row_and_sorted(score, tmp_path, monkeypatch):
    """A call whose rows would be sorted, in scratch for a chunk of a few hundred rows, whose sort's arrays alone are
    larger: shorter chunks, which are not sorted, and the same bits. 1024 experts: 0.3 MB of sorts' arrays; 60 000 rows,
    past the 58 594 from which a sort pays at n = 64."""
    import torch
    from yggdrasil_amd import _lib
    from yggdrasil_amd.inference import Yggdrasil
    monkeypatch.setenv("YGG_SCAN", "1")
    p = tmp_path / "m.bin"
    synth.write_model(K(64, 16, 10, 27, 3, 8, 16), 6, p)
    m, lib = Yggdrasil.load(p), _lib.lib()
    B, T = 60, 1000
    x = torch.tensor(np.random.default_rng(7).integers(0, 27, (B, T + 1)), dtype=torch.int32, device=m.device)
    xd, yd = x[:, :-1].contiguous(), x[:, 1:].contiguous()
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    q = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    least, whole = lib.ygg_scratch(m._h, 60, 2, score), lib.ygg_scratch(m._h, B, T, score)
    got = []
    for size in (None, least, least + 100_000, least + 250_000, least + 400_000, whole - 256, whole):
        st, nll = m.init_state(B), torch.zeros(B, dtype=torch.float64, device=m.device)
        lg = torch.zeros(B, T, 27, device=m.device)
        ws = None if size is None else torch.empty(size, dtype=torch.uint8, device=m.device)
        if score and size is None:
            rc = lib.ygg_score(m._h, ptr(xd), ptr(yd), B, T, ptr(st), ptr(nll), q)
        elif score:
            rc = lib.ygg_score_scratch(m._h, ptr(xd), ptr(yd), B, T, ptr(st), ptr(nll), ptr(ws), size, q)
        elif size is None:
            rc = lib.ygg_run(m._h, ptr(xd), B, T, ptr(st), ptr(lg), None, None, None, q)
        else:
            rc = lib.ygg_run_scratch(m._h, ptr(xd), B, T, ptr(st), ptr(lg), None, ptr(ws), size, q)
        assert rc == 0, f"scratch of {size} bytes: {lib.ygg_last_error().decode()}"
        got.append([t.cpu().numpy() for t in (st, nll, lg)])
        for a, b in zip(got[0], got[-1]):
            np.testing.assert_array_equal(a, b)
    m.close()


def test_scan_taken_where_it_pays(tmp_path, monkeypatch):
    """The calls that go layer by layer: long enough ones of few streams, large batches of the trained shapes and all but
    the shortest factored calls, but no call of one token, no short one of a table model and none with a kernel forced."""
    from yggdrasil_amd import _lib
    from yggdrasil_amd.inference import Yggdrasil
    p, f = tmp_path / "m.bin", tmp_path / "f.bin"
    synth.write_model(K(128, 16, 10, 27, 5, 16, 32), 7, p)
    synth.write_model(K(128, 16, 10, 27, 5, 16, 32, input_rank=32), 7, f)
    lib = _lib.lib()
    m, mf = Yggdrasil.load(p), Yggdrasil.load(f)
    takes = lambda m, B, T: lib.ygg_scratch(m._h, B, T, 0) > 0  # noqa: E731
    assert takes(m, 1, 1024) and takes(m, 4096, 256) and takes(mf, 1, 16) and takes(mf, 4096, 64)
    assert not takes(m, 1, 1) and not takes(m, 1, 16) and not takes(m, 256, 32) and not takes(mf, 8, 1)
    m.close()
    mf.close()
    # short calls of few layers stay token by token at any number of streams (us token by token / layer by layer: 4096 x 2
    # tokens of the two 128-wide layers 13 / 87, 256 x 8 18 / 24, 256 x 4 of the factored ones 18 / 27)
    for spec, no, yes in ((K(128, 16, 12, 32, 2, 8, 16), ((1, 2), (4096, 2), (256, 8), (1500, 16)), ((1, 256), (64, 256))),
                          (K(64, 16, 6, 64, 2, 8, 16, input_rank=32), ((1, 2), (256, 4), (4096, 6)), ((1, 16), (64, 64))),
                          (K(256, 16, 5, 27, 2, 32, 64), ((1, 4), (4096, 4), (700, 12)), ((4, 48), (64, 64)))):
        synth.write_model(spec, 7, p)
        m = Yggdrasil.load(p)
        for B, T in no:
            assert not takes(m, B, T) and not lib.ygg_scratch(m._h, B, T, 1), (spec, B, T)
        for B, T in yes:
            assert takes(m, B, T) and lib.ygg_scratch(m._h, B, T, 1) and lib.ygg_scratch(m._h, B, T, 2), (spec, B, T)
        m.close()
    monkeypatch.setenv("YGG_KERNEL", "fast")
    m = Yggdrasil.load(p)
    assert not takes(m, 1, 1024)
    m.close()
