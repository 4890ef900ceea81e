"""Every binary layer of a 32x32 patch in one kernel (bnn_tail.hip), for v1 and
stem models of at most 16, 32, 64, 128, 256 channels at the five levels, with
1 or 2 patches a block by the launch's size.  BNN_TAIL=0 keeps the layers
apart; the logits are the same bit for bit, and the checker's."""
import numpy as np
import pytest

from bnns_to_c_amd import blob as B
from bnns_to_c_amd import engine as E
from bnns_to_c_amd import synth

pytestmark = pytest.mark.gpu


def _pair(tmp_path, monkeypatch, b):
    p = tmp_path / "m.blob"
    p.write_bytes(B.to_bytes(b))
    cls = E.StemEngine if b.version == B.VERSION_STEM else E.Engine
    monkeypatch.delenv("BNN_TAIL", raising=False)
    one = cls(str(p))
    monkeypatch.setenv("BNN_TAIL", "0")
    apart = cls(str(p))
    monkeypatch.delenv("BNN_TAIL")
    return one, apart


def _ops(eng, x):
    """label -> profiler op name of one forward."""
    E.prof_reset()
    E.prof_enable(True)
    try:
        eng.forward_batch(x)
    finally:
        E.prof_enable(False)
    return {lab: op for lab, op, _ms, _w in E.prof_records()}


def _takes(one, apart, x):
    """The first model runs its layers as one kernel, the second apart."""
    assert "bconv_tail" in _ops(one, x).values()
    assert "enc1.c2" in _ops(apart, x)


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


# one patch, a few, a partial last block of two, more than a round
@pytest.mark.parametrize("base,N,cov", [(16, 1, False), (16, 5, True), (16, 301, False), (16, 515, True),
                                         (16, 1031, True), (8, 2, True), (12, 3, True), (4, 1, True), (8, 601, False)])
def test_tail_equals_layers(tmp_path, monkeypatch, orc, base, N, cov):
    b = synth.make_blob(seed=90 + base + N, base=base, coverage=cov)
    one, apart = _pair(tmp_path, monkeypatch, b)
    x = synth.make_input(91 + N, N, 120, 32, 32)
    _takes(one, apart, x)
    got = one.forward_batch(x)
    assert np.array_equal(_bits(got), _bits(apart.forward_batch(x)))
    model = orc.parse(B.to_bytes(b))
    for n in {0, N // 2, N - 1}:
        assert np.array_equal(_bits(got[n]), _bits(model.forward(x[n]))), n
    one.close()
    apart.close()


@pytest.mark.parametrize("base,stem,N", [(16, 16, 1), (16, 16, 700), (8, 8, 5), (16, 12, 300)])
def test_tail_stem(tmp_path, monkeypatch, base, stem, N):
    b = synth.make_blob_v2(seed=92 + N, base=base, stem=stem, coverage=True)
    one, apart = _pair(tmp_path, monkeypatch, b)
    x = synth.make_input(93 + N, N, 120, 32, 32)
    _takes(one, apart, x)
    assert np.array_equal(_bits(one.forward_batch(x)), _bits(apart.forward_batch(x)))
    one.close()
    apart.close()


@pytest.mark.parametrize("H,W,classes", [(70, 100, 3), (33, 300, 5), (300, 290, 1)])
def test_tail_scene(tmp_path, monkeypatch, H, W, classes):
    """Edge patches past the scene, other class counts."""
    b = synth.make_blob(seed=94, base=16, n_classes=classes, coverage=True)
    one, apart = _pair(tmp_path, monkeypatch, b)
    _takes(one, apart, synth.make_input(98, 2, 120, 32, 32))
    cube = np.random.default_rng(95).standard_normal((120, H, W), dtype=np.float32)
    assert np.array_equal(_bits(one.forward_patched(cube, 32)), _bits(apart.forward_patched(cube, 32)))
    one.close()
    apart.close()


@pytest.mark.parametrize("base,H,W", [(20, 32, 32), (16, 33, 32), (16, 32, 31), (16, 64, 64)])
def test_tail_not_taken(tmp_path, monkeypatch, base, H, W):
    """A model just too wide, and patches of other sizes, run their layers apart."""
    one, apart = _pair(tmp_path, monkeypatch, synth.make_blob(seed=96, base=base))
    x = synth.make_input(97, 2, 120, H, W)
    assert "enc1.c2" in _ops(one, x)
    one.close()
    apart.close()
