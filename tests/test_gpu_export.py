"""GPU signed LEB128 (sft_leb128_encode) and the .nnue FT section against the
oracle: identical bytes; full-size weights through a decode round trip."""

import numpy as np
import pytest
import torch

from gpu_helpers import DEV, announce, dev, host
from oracle import ft_oracle
from oracle import leb128_oracle as leb
from sft_amd import _native
from src.model.modules.features import get_feature_cls
from src.model.quantize import QuantizationConfig, QuantizationManager
from src.scripts.serialize import FeatureTransformerWriter

pytestmark = pytest.mark.gpu

LIMITS = {np.int8: [0, 1, -1, 63, 64, -64, -65, 127, -128],
          np.int16: [0, 1, -1, 63, 64, -64, -65, 8191, 8192, -8192, -8193, 32767, -32768],
          np.int32: [0, 1, -1, 8191, 8192, -8193, 1048575, -1048576, 2**31 - 1, -2**31]}


@pytest.mark.parametrize("dtype,n", [(np.int8, 1), (np.int8, 5000), (np.int16, 4097), (np.int16, 100003),
                                     (np.int32, 77777)])
def test_leb128_matches_oracle(dtype, n):
    announce(f"leb128 {dtype.__name__} n={n}")
    g = np.random.default_rng(n)
    info = np.iinfo(dtype)
    a = g.integers(info.min, info.max + 1, n, dtype=np.int64).astype(dtype)
    small = g.integers(-300, 300, n).astype(dtype)
    a = np.where(g.random(n) < 0.7, small, a)
    a[:min(n, len(LIMITS[dtype]))] = LIMITS[dtype][:min(n, len(LIMITS[dtype]))]
    got = host(_native.leb128_encode(dev(a))).tobytes()
    assert got == leb.encode(a)


# tiles of 4096 values, groups of 4 tiles; views off the 16-byte alignment
@pytest.mark.parametrize("dtype", [np.int8, np.int16, np.int32])
@pytest.mark.parametrize("n", [15, 16, 17, 4095, 4096, 16383, 16384, 16385, 40961])
@pytest.mark.parametrize("skip", [0, 1, 3])
def test_leb128_tile_edges(dtype, n, skip):
    announce(f"leb128 edges {dtype.__name__} n={n} skip={skip}")
    g = np.random.default_rng(n + skip)
    info = np.iinfo(dtype)
    a = (g.integers(info.min, info.max + 1, n + skip) >> g.integers(0, 8 * info.dtype.itemsize, n + skip)).astype(dtype)
    assert host(_native.leb128_encode(dev(a)[skip:])).tobytes() == leb.encode(a[skip:])


def test_leb128_scanned_groups():
    """More groups than a writing workgroup sums itself (8192 of 16 384 values)."""
    announce("leb128 scanned groups")
    n = 8192 * 16384 + 5
    a = torch.randint(-64, 64, (n,), dtype=torch.int8, device=DEV)  # codes of one byte
    a[7], a[n - 2] = 100, -100                                       # and two of two
    got = _native.leb128_encode(a)
    assert got.numel() == n + 2
    one = a & 0x7F
    assert torch.equal(got[:7].to(torch.int8), one[:7]) and host(got[7:9]).tobytes() == bytes([0xE4, 0x00])
    assert torch.equal(got[9:n - 1].to(torch.int8), one[8:n - 2])
    assert host(got[n - 1:n + 1]).tobytes() == bytes([0x9C, 0x7F]) and int(got[-1]) == int(one[-1])


@pytest.mark.parametrize("n", [1, 7, 8, 9, 2049, 100003])
@pytest.mark.parametrize("skip", [0, 1])
def test_quantize_run_edges(n, skip):
    announce(f"quantize n={n} skip={skip}")
    g = np.random.default_rng(n)
    x = (g.standard_normal(n + skip) * 200).astype(np.float32)
    x[-1] = np.float32(0.5 / 255.0)
    got = host(_native.quantize_i16(dev(x)[skip:], 255.0))
    assert np.array_equal(got, ft_oracle.quantize_i16(x[skip:], 255.0))


def test_leb128_empty():
    assert _native.leb128_encode(torch.zeros(0, dtype=torch.int16, device=DEV)).numel() == 0


def test_leb128_full_size_round_trip():
    announce("leb128 22528 x 1040 int16 round trip")
    g = np.random.default_rng(5)
    a = np.clip(np.rint(g.standard_normal((22528, 1040)) * 40), -32768, 32767).astype(np.int16)
    a[0, :4] = [32767, -32768, 8192, -8193]
    buf = host(_native.leb128_encode(dev(a))).tobytes()
    assert np.array_equal(leb.decode(buf, a.size), a.reshape(-1).astype(np.int64))


@pytest.mark.parametrize("name,l1", [("HalfKAv2_hm^", 64), ("Full_Threats+HalfKAv2_hm^", 32)])
def test_ft_section_matches_oracle(name, l1):
    announce(f"nnue FT section {name} L1={l1}")
    torch.manual_seed(2)
    ft = get_feature_cls(name)(l1 + 8).to(DEV)
    with torch.no_grad():
        for f in ft.features:
            f.weight.uniform_(-0.4, 0.4)  # within int8 after the 255 scale (threat rows are int8)
            if hasattr(f, "virtual_weight"):
                f.virtual_weight.uniform_(-0.05, 0.05)
        ft.bias.uniform_(-0.5, 0.5)
    q = QuantizationManager(QuantizationConfig())
    got = bytes(FeatureTransformerWriter(ft, l1, q).buf)
    blocks = [(int(f.NUM_REAL_FEATURES), "int8" if f.EXPORT_WEIGHT_DTYPE == torch.int8 else "int16")
              for f in ft.features]
    want = leb.ft_section(ft.HASH, l1, host(ft.bias), host(ft.get_export_weights()), blocks, q.ft_quantized_one,
                          q.psqt_scale)
    assert got == want


@pytest.mark.parametrize("name,l1,mode", [("HalfKAv2_hm^", 64, "layer"), ("Full_Threats+HalfKAv2_hm^", 32, "moe"),
                                          ("HalfKAv2_hm^", 32, "none")])
def test_whole_nnue_file(name, l1, mode):
    """The whole file with the FT section written on the GPU: its FT bytes are
    the oracle's, and the header, router and FC buckets parse back to the
    quantized layers (tests/test_nnue_writer_cpu.py checks the same layout with
    the CPU FT section)."""
    from nnue_model import Model
    from test_nnue_writer_cpu import _check_file
    from src.scripts.serialize import NNUEWriter

    announce(f"whole .nnue {name} L1={l1} {mode}")
    m = Model(name, L1=l1, count=8, stacks="none" if mode == "none" else "layer", moe=mode == "moe", device=DEV)
    buf = bytes(NNUEWriter(m, description="gpu").buf)
    _check_file(m, buf, mode)
    blocks = [(int(f.NUM_REAL_FEATURES), "int8" if f.EXPORT_WEIGHT_DTYPE == torch.int8 else "int16")
              for f in m.input.features]
    q = m.quantization
    want_ft = leb.ft_section(m.input.HASH, l1, host(m.input.bias), host(m.input.get_export_weights()), blocks,
                             q.ft_quantized_one, q.psqt_scale)
    assert buf[12 + 3:12 + 3 + len(want_ft)] == want_ft
