"""Host tokens are checked against [0, vocab) whatever their integer type (yggdrasil_amd.inference.host_tokens), as the
reference rejects a bad token file up front (cpu/ygg.cpp:493-495); and the calls that take them refuse what it refuses."""
import numpy as np
import pytest
import torch

from yggdrasil_amd import synth
from yggdrasil_amd.inference import Yggdrasil, device_tokens, host_tokens

TYPES = ["int8", "uint8", "int16", ">i2", "uint16", "int32", ">i4", "uint32", "int64", ">i8", "uint64"]


@pytest.mark.parametrize("vocab", [1, 5, 127, 128, 129, 200, 256, 300])
@pytest.mark.parametrize("dtype", TYPES)
def test_range_check_over_types(dtype, vocab):
    info = np.iinfo(dtype)
    ok = sorted({0, min(vocab // 2, info.max), min(vocab - 1, info.max)})
    for a in (np.array(ok, dtype), np.array([ok, ok], dtype)[:, ::-1], np.array(ok[-1], dtype), np.zeros((0, 3), dtype)):
        got = host_tokens(a, vocab)
        assert got.dtype.kind in "iu" and got.shape == a.shape
        np.testing.assert_array_equal(got.astype(np.int64), a.astype(np.int64))
    for bad in {-1, -2, -100, -128, info.min, vocab, vocab + 1, info.max}:
        if not info.min <= bad <= info.max or 0 <= bad < vocab:
            continue
        for a in (np.array([0, bad, 0], dtype), np.array([[0, 0], [bad, 0]], dtype).T, np.array(bad, dtype)):
            with pytest.raises(ValueError, match="out of range"):
                host_tokens(a, vocab)
            with pytest.raises(ValueError, match="out of range"):
                device_tokens(a, vocab, torch.device("cuda", 0))
            if a.dtype.isnative and a.dtype.kind == "i":
                with pytest.raises(ValueError, match="out of range"):
                    host_tokens(torch.from_numpy(np.ascontiguousarray(a)), vocab)


@pytest.mark.parametrize("a", [np.zeros(3), np.zeros(3, bool), [0.5], ["a"]], ids=["f8", "bool", "list", "text"])
def test_no_integers(a):
    with pytest.raises(ValueError, match="integers"):
        host_tokens(a, 256)


@pytest.mark.parametrize("targets", [False, True])
def test_score_takes_windows_of_two_axes(targets):
    """Before any device is touched; a third axis was once read as more of the first rows' tokens."""
    m = object.__new__(Yggdrasil)
    a = np.zeros((2, 3, 4), np.int64)
    with pytest.raises(ValueError, match="tokens must be"):
        m.score(a, targets=a if targets else None)


@pytest.mark.gpu
def test_calls_refuse_narrow_negative_tokens(tmp_path):
    """run, step and score on int8 arrays, whose -1 has the bits of token 255; the same values as other types pass."""
    p = tmp_path / "m.bin"
    synth.write_model(synth.ModelSpec(64, 16, 4, 256, 2, 8, 16), 3, p)
    m = Yggdrasil.load(p)
    good = np.arange(36).reshape(4, 9) % 128
    bad = good.astype(np.int8)
    bad[2, 5] = -1
    for call in (lambda a: m.run(a), lambda a: m.step(a[2], m.init_state(9)), lambda a: m.score(a),
                 lambda a: m.score(good, targets=a), lambda a: m.score(a, targets=good), lambda a: m.generate(a, 2)):
        with pytest.raises(ValueError, match="out of range"):
            call(bad)
    for t in ("int8", "uint8", "int16", "uint64"):
        np.testing.assert_array_equal(m.score(good.astype(t)), m.score(good))
        assert torch.equal(m.run(good.astype(t))["logits"], m.run(good)["logits"])
    m.close()
