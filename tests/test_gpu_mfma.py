"""The binary 3x3 conv on the matrix cores (bnn_bconv_mfma.hip).

The kernel computes the same P as csrc/bnn_conv.c:23-36 (P = 2*D - S with
D the FP4 product of 0/1 activations and +-1 weights, S the weight sum over
the in-image taps), with the rule and the 2x2 max-pool of
csrc/bnn_fold.c:37-60 and csrc/bnn_maxpool.c:28-48 fused.  BNN_BCONV_MFMA=2
routes every conv through it; every stage of the forward must then equal the
checker's bit for bit, as on the popcount path.  The default rule is checked
on the wide layers that it names and on both sides of its lines, and the
isolated layer entry point must agree with the popcount kernel.
"""
import numpy as np
import pytest

from bnns_to_c_amd import blob as B
from bnns_to_c_amd import engine as E
from bnns_to_c_amd import synth

pytestmark = pytest.mark.gpu


def _same(a, b):
    a, b = np.asarray(a), np.asarray(b)
    if a.shape != b.shape or a.dtype != b.dtype:
        return False
    if a.dtype == np.float32:
        return np.array_equal(a.view(np.uint32), b.view(np.uint32))
    return np.array_equal(a, b)


def _ops(eng, x):
    """label -> profiler op name of one forward."""
    E.prof_reset()
    E.prof_enable(True)
    try:
        eng.forward_batch(x)
    finally:
        E.prof_enable(False)
    return {lab: op for lab, op, _ms, _w in E.prof_records()}


def _check_stages(eng, model, x):
    logits, st = eng.forward_debug(x)
    for n in range(x.shape[0]):
        want, ref_st = model.forward(x[n], stages=True)
        for name, arr in st.items():
            if name == "logits":
                continue
            assert _same(arr[n], ref_st[name]), (name, n)
        assert _same(logits[n], want), n


# (seed, base, N, H, W): patches of several tiles (64x64, 96x64 and its
# 48x32 level), whole-patch tiles with a partial last tile (8x8 levels, N
# odd), an odd number of input words (base 24: 96 -> 192 channels at 8x8),
# rows wider than 64 in tiles of 32 columns (base 64 at 64x256: levels 256
# and 128 wide, with pools and concats, and a 4x16 bottleneck in tiles of
# four whole patches)
@pytest.mark.parametrize("seed,base,N,H,W", [
    (21, 32, 2, 64, 64),
    (22, 32, 3, 32, 32),
    (23, 16, 3, 32, 32),
    (24, 24, 1, 64, 64),
    (25, 32, 1, 96, 64),
    (26, 64, 1, 64, 256),
])
def test_forced_mfma_stages_vs_checker(tmp_path, orc, monkeypatch, seed, base, N, H, W):
    monkeypatch.setenv("BNN_BCONV_MFMA", "2")
    monkeypatch.setenv("BNN_MID", "0")  # the fused middle would take base 16's matrix-core layers
    b = synth.make_blob(seed=seed, base=base)
    p = tmp_path / "m.blob"
    p.write_bytes(B.to_bytes(b))
    eng = E.Engine(str(p))
    x = synth.make_input(seed + 100, N, 120, H, W)
    ops = _ops(eng, x)
    assert any(op.endswith("_mfma") for op in ops.values()), ops
    _check_stages(eng, orc.parse(B.to_bytes(b)), x)
    eng.close()


def test_default_rule_picks_by_size(tmp_path, orc, monkeypatch):
    """Default: each layer on its faster kernel (mfma_conv_pays); a layer's op
    names the kernel that ran.  One image: the deep layers on the matrix cores,
    shallow folds, which fill no launch, on the popcount kernel; 64 patches:
    every layer on the matrix cores."""
    monkeypatch.delenv("BNN_BCONV_MFMA", raising=False)
    b = synth.make_blob(seed=26, base=32)
    p = tmp_path / "m.blob"
    p.write_bytes(B.to_bytes(b))
    eng = E.Engine(str(p))
    x = synth.make_input(126, 1, 120, 128, 128)
    took = {lab for lab, op in _ops(eng, x).items() if op.endswith("_mfma")}
    assert {"enc4.c2", "bott.c2", "dec4.c1"} <= took, took
    assert not took & {"enc1.c2", "enc2.c1", "enc3.c1", "enc4.c1", "dec3.c2", "dec2.c2", "dec1.c2"}, took
    _check_stages(eng, orc.parse(B.to_bytes(b)), x)
    ops = _ops(eng, synth.make_input(127, 64, 120, 128, 128))
    assert all(op.endswith("_mfma") for lab, op in ops.items() if lab not in ("enc1.conv1", "dec1.c2")), ops
    eng.close()


@pytest.mark.parametrize("N,H,W,c", [(1024, 32, 32, 128), (5, 8, 8, 64), (3, 16, 16, 256), (2, 64, 64, 64),
                                     (2, 32, 128, 64), (1, 16, 256, 128)])
def test_layer_fold_pool_matches_popcount(monkeypatch, N, H, W, c):
    import torch
    a = synth.make_bits(40 + c, N, H, W, c)
    w = synth.make_signs(41, c, c)
    t1 = synth.make_thresholds(42, c, c * 9 // 4)
    t2 = synth.make_thresholds(43, c, c * 9 // 4)
    da = torch.from_numpy(a).cuda()
    act = torch.empty((N, H, W, c // 32), dtype=torch.int32, device="cuda")
    E.pack_act_device(da.data_ptr(), act.data_ptr(), N, c, H, W, None)
    torch.cuda.synchronize()
    outs = {}
    for mode in ("0", "2"):
        monkeypatch.setenv("BNN_BCONV_MFMA", mode)
        L = E.ConvLayer(B.pack_kidx(w), c, c, t1, t2)
        skip = torch.full((N, H, W, c // 32), -1, dtype=torch.int32, device="cuda")
        down = torch.full((N, H // 2, W // 2, c // 32), -1, dtype=torch.int32, device="cuda")
        L.fold_pool_device(act.data_ptr(), N, H, W, skip.data_ptr(), down.data_ptr(), None)
        torch.cuda.synchronize()
        outs[mode] = (skip.cpu().numpy(), down.cpu().numpy())
        L.close()
    assert np.array_equal(outs["0"][0], outs["2"][0])
    assert np.array_equal(outs["0"][1], outs["2"][1])


def _act(torch, seed, N, H, W, c):
    """Random packed bits, the unused high bits of the last word 0."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    a = torch.randint(-2**31, 2**31, (N, H, W, (c + 31) // 32), generator=g, device="cuda", dtype=torch.int64)
    a = a.to(torch.int32)
    if c % 32:
        a[..., -1] &= (1 << c % 32) - 1
    return a


# tiles of whole patches (1 to 64 of them, a partial last one), of whole rows
# (odd widths and heights, an even split), of columns (67, 130 wide); one to
# four tiles staged together; paired taps (16 and fewer channels); 1 to 12
# input words, planes of four with a remainder; channel groups of 16, 32 and
# 64 with a partial last one; weights kept in LDS and streamed through it
SHAPES = [(700, 2, 2, 256, 256), (9, 5, 3, 40, 24), (37, 4, 4, 384, 128), (3, 13, 9, 40, 96), (2, 33, 47, 8, 16),
          (5, 45, 51, 24, 24), (2, 64, 67, 96, 48), (1, 31, 130, 72, 160), (1100, 32, 32, 16, 16),
          (70, 64, 64, 32, 32), (1, 7, 200, 200, 72), (400, 8, 8, 64, 64), (1, 1, 1, 33, 7), (3, 3, 64, 129, 65)]


@pytest.mark.parametrize("N,H,W,cin,cout", SHAPES)
def test_layer_shapes_match_popcount(monkeypatch, N, H, W, cin, cout):
    """P, skip bits and pooled bits of an isolated layer: the matrix cores
    against the popcount kernel, every rule type, bit for bit."""
    import torch
    act = _act(torch, 50 + cin, N, H, W, cin)
    w = B.pack_kidx(synth.make_signs(51, cout, cin))
    r1 = synth.make_rules(52, cout, cin * 9, coverage=True)
    r2 = synth.make_rules(53, cout, cin * 9, coverage=True)
    cwo = (cout + 31) // 32
    outs = {}
    for mode in ("0", "2"):
        monkeypatch.setenv("BNN_BCONV_MFMA", mode)
        L = E.ConvLayer(w, cin, cout, r1, r2)
        P = torch.full((N, cout, H, W), -7, dtype=torch.int32, device="cuda")
        L.P_device(act.data_ptr(), N, H, W, P.data_ptr(), None)
        got = [P]
        if H >= 2 and W >= 2:
            skip = torch.full((N, H, W, cwo), -1, dtype=torch.int32, device="cuda")
            down = torch.full((N, H // 2, W // 2, cwo), -1, dtype=torch.int32, device="cuda")
            only = torch.full((N, H // 2, W // 2, cwo), -1, dtype=torch.int32, device="cuda")
            L.fold_pool_device(act.data_ptr(), N, H, W, skip.data_ptr(), down.data_ptr(), None)
            L.fold_pool_device(act.data_ptr(), N, H, W, None, only.data_ptr(), None)
            got += [skip, down, only]
        torch.cuda.synchronize()
        outs[mode] = [t.cpu().numpy() for t in got]
        L.close()
    for a, b in zip(outs["0"], outs["2"]):
        assert np.array_equal(a, b)


# both sides of the default rule's lines: P by depth, row length and pixels,
# pools by depth and size
@pytest.mark.parametrize("N,H,W,cin,cout", [(5220, 10, 5, 56, 32), (70, 64, 64, 64, 64), (60, 64, 64, 64, 64),
                                            (300, 31, 41, 104, 24), (60, 31, 41, 104, 24), (246, 6, 17, 368, 56),
                                            (7, 22, 20, 248, 176), (14, 22, 20, 248, 176), (45, 33, 93, 80, 24),
                                            (45, 33, 93, 88, 24), (2, 49, 7, 96, 40)])
def test_default_rule_layers_match_popcount(monkeypatch, N, H, W, cin, cout):
    import torch
    act = _act(torch, 55, N, H, W, cin)
    w = B.pack_kidx(synth.make_signs(56, cout, cin))
    r1 = synth.make_rules(57, cout, cin * 9, coverage=True)
    r2 = synth.make_rules(58, cout, cin * 9, coverage=True)
    cwo = (cout + 31) // 32
    outs = {}
    for mode in ("0", "1"):
        monkeypatch.setenv("BNN_BCONV_MFMA", mode)
        L = E.ConvLayer(w, cin, cout, r1, r2)
        P = torch.full((N, cout, H, W), -7, dtype=torch.int32, device="cuda")
        skip = torch.full((N, H, W, cwo), -1, dtype=torch.int32, device="cuda")
        down = torch.full((N, H // 2, W // 2, cwo), -1, dtype=torch.int32, device="cuda")
        L.P_device(act.data_ptr(), N, H, W, P.data_ptr(), None)
        L.fold_pool_device(act.data_ptr(), N, H, W, skip.data_ptr(), down.data_ptr(), None)
        torch.cuda.synchronize()
        outs[mode] = [t.cpu().numpy() for t in (P, skip, down)]
        L.close()
    for a, b in zip(outs["0"], outs["1"]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("base,N,H,W", [(8, 3, 35, 41), (16, 2, 32, 32), (24, 2, 45, 51), (20, 1, 70, 83)])
def test_forced_forward_vs_checker(tmp_path, orc, monkeypatch, base, N, H, W):
    """Whole forwards with every layer on the matrix cores (the concat layers
    with an upsample that leaves odd edges uncovered, the head): every stage
    against the checker."""
    monkeypatch.setenv("BNN_BCONV_MFMA", "2")
    monkeypatch.setenv("BNN_MID", "0")
    b = synth.make_blob(seed=60 + base, base=base, coverage=True)
    p = tmp_path / "m.blob"
    p.write_bytes(B.to_bytes(b))
    eng = E.Engine(str(p))
    _check_stages(eng, orc.parse(B.to_bytes(b)), synth.make_input(160, N, 120, H, W))
    eng.close()
