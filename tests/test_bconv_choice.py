"""Which kernel a binary conv takes by default (mfma_conv_pays,
bnns_to_c_amd/csrc/bnn_bconv_mfma.hip): layers that measured at least a tenth
faster on one of the two, on either side of the choice.  CPU only: the choice
is host code."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
LIB = os.path.join(ROOT, "bnns_to_c_amd", "lib")

# (epilogue, cin, cout, skip channels of a concat, N, H, W, popcount us, matrix-core us)
LAYERS = [
    ("pool", 16, 16, 0, 1618, 70, 25, 31.1, 45.1),
    ("pool", 16, 8, 0, 35609, 9, 17, 39.5, 101.7),
    ("pool", 32, 8, 0, 6154, 15, 19, 17.1, 39.2),
    ("pool", 16, 16, 0, 3444, 13, 48, 23.9, 39.7),
    ("pool", 16, 72, 0, 3013, 26, 8, 33.0, 37.2),
    ("pool", 40, 192, 0, 192, 35, 4, 16.1, 10.1),
    ("pool", 128, 128, 0, 1024, 32, 32, 288.0, 82.0),
    ("pool", 152, 16, 0, 7466, 29, 6, 66.9, 47.4),
    ("fold", 64, 64, 0, 1, 128, 128, 5.0, 7.1),
    ("fold", 96, 192, 0, 1, 32, 32, 5.2, 8.1),
    ("fold", 192, 64, 64, 3, 32, 32, 7.0, 10.1),
    ("fold", 48, 16, 16, 61, 113, 73, 12.7, 16.9),
    ("fold", 64, 64, 0, 1, 145, 32, 5.2, 7.0),
    ("fold", 512, 512, 0, 1, 32, 32, 33.8, 12.4),
    ("fold", 256, 256, 0, 148, 4, 4, 16.4, 10.5),
    ("fold", 384, 384, 0, 48, 2, 3, 14.0, 11.5),
    ("fold", 256, 512, 0, 155, 1, 5, 17.0, 11.2),
    ("fold", 768, 256, 256, 13, 2, 3, 14.6, 16.6),
    ("fold", 1152, 384, 384, 1, 13, 20, 38.6, 21.4),
    ("fold", 768, 256, 256, 1, 17, 36, 26.4, 16.4),
    ("head", 32, 32, 0, 64, 256, 256, 97.6, 69.1),
    ("head", 24, 24, 0, 152, 113, 51, 28.2, 34.0),
    ("P", 64, 64, 0, 256, 64, 64, 89.0, 75.0),
    ("P", 72, 168, 0, 2381, 17, 5, 67.1, 91.3),
]


def _build(tmp_path, source):
    assert os.path.exists(os.path.join(LIB, "libbnn_hip.so")), "the library is not built"
    exe = tmp_path / "check"
    subprocess.run([HIPCC, "-O1", "-std=c++17", "-I", os.path.join(ROOT, "bnns_to_c_amd", "csrc"), "-I",
                    os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", source), "-o", str(exe),
                    "-L", LIB, "-lbnn_hip", "-Wl,-rpath," + LIB], check=True, capture_output=True, timeout=300)
    return str(exe)


def _choice(tmp_path, layers):
    """[(taken by default, fits)] of (epilogue, cin, cout, skip, N, H, W)."""
    text = "".join("%s %d %d %d %d %d %d\n" % layer for layer in layers)
    r = subprocess.run([_build(tmp_path, "bconv_choice_check.cpp")], input=text, capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    out = [tuple(map(int, line.split())) for line in r.stdout.splitlines()]
    assert len(out) == len(layers)
    return out


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc (for the HIP headers) not found")
def test_layers_take_their_faster_kernel(tmp_path):
    took = _choice(tmp_path, [layer[:7] for layer in LAYERS])
    wrong = [layer for layer, t in zip(LAYERS, took) if t[0] != int(layer[8] < layer[7])]
    assert not wrong, wrong


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc (for the HIP headers) not found")
def test_gpu_shapes_fit(tmp_path):
    """The layers that the GPU tests force onto the matrix cores run there."""
    from test_gpu_mfma import SHAPES
    layers = [(epi, cin, cout, 0, N, H, W) for N, H, W, cin, cout in SHAPES for epi in ("P", "pool")]
    assert all(fits for _, fits in _choice(tmp_path, layers))


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc (for the HIP headers) not found")
def test_pad_pixel_concat_is_refused(tmp_path):
    """1: hipErrorInvalidValue."""
    r = subprocess.run([_build(tmp_path, "bconv_refusal_check.cpp")], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.split() == ["1"], r.stdout + r.stderr
