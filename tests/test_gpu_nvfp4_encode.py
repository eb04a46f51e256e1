"""The loader's NVFP4 conversions on the device at the edges of their kernels: the f16 weight
quantizer (whole and partial blocks, aligned and not) and the in-place row-to-tiled repack (fewer
rows of pieces than threads, exactly the register limit, one tile past it). Whole bytes: exact."""
import sys

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _bits(rng, n):
    """f16 patterns of every kind: ordinary, groups of zeros, subnormals, infinities, NaNs."""
    w = (rng.standard_normal(n) * 0.02).astype(np.float16).view(np.uint16)
    if n >= 256:
        w[:32] = 0
        w[32:64] = rng.integers(0, 2, 32) * 0x8000
        w[64:96] = rng.integers(1, 0x400, 32)
        w[96:128:3] = 0x7C00
        w[128:160:5] = 0x7E01
        w[160:192] = 0xFE00
        # any pattern but signalling NaNs: the host's f16 conversion keeps those signalling, so the
        # oracle's maximum takes them otherwise than the device's (either kernel's) does
        any_ = rng.integers(0, 65536, 64)
        w[192:256] = np.where((any_ & 0x7FFF) > 0x7C00, any_ | 0x200, any_)
    return w


@pytest.mark.parametrize("m,k,shift", [(1, 32, 0), (1, 64, 0), (3, 32, 0), (16, 512, 0), (257, 32, 0),
                                       (31, 1056, 0), (5, 96, 1), (64, 4096, 1)])
def test_weight_quantizer(m, k, shift):
    """shift = 1: input and codes 2 and 1 bytes past an aligned address."""
    from vib3_amd import _lib
    _say(f"case: weight quantizer m={m} k={k} shift={shift}")
    w = _bits(np.random.default_rng(m * k), m * k)
    src = torch.zeros(m * k + shift, dtype=torch.int16, device="cuda")
    src[shift:] = torch.from_numpy(w.view(np.int16)).cuda()
    data = torch.full((m * k // 2 + 1 + 64,), 0xA5, dtype=torch.uint8, device="cuda")
    sc = torch.full((m * k // 32 + 8,), 0x5A5A, dtype=torch.int16, device="cuda")
    _lib.call("vib3_launch_fp16_to_nvfp4_weight", src.data_ptr() + 2 * shift, data.data_ptr() + shift,
              sc.data_ptr(), m, k, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    rd, rs = O.fp16_to_nvfp4_weight(w, m, k)
    d, s = data.cpu().numpy(), sc.cpu().numpy().view(np.uint16)
    assert np.array_equal(d[shift:shift + m * k // 2], rd)
    assert np.array_equal(s[:m * k // 32], rs)
    assert (d[shift + m * k // 2:] == 0xA5).all() and (s[m * k // 32:] == 0x5A5A).all()


@pytest.mark.parametrize("m,k,shift", [(63, 4160, 0), (64, 4096, 0), (257, 1056, 0), (2, 131104, 0), (64, 4096, 1)])
def test_weight_quantizer_kernel_choice(m, k, shift):
    """Matrices just below and above the size from which a lane takes eight weights, with whole and
    partial last blocks."""
    test_weight_quantizer(m, k, shift)


@pytest.mark.parametrize("m,k", [(16, 64), (48, 192), (16, 2048), (32, 2112), (16, 16384), (16, 16448)])
def test_repack_row_to_tiled(m, k):
    from vib3_amd import kernels as K
    _say(f"case: repack m={m} k={k}")
    row = np.random.default_rng(k).integers(0, 256, m * k // 2, dtype=np.uint8)
    buf = torch.full((m * k // 2 + 64,), 0xA5, dtype=torch.uint8, device="cuda")
    buf[:m * k // 2] = torch.from_numpy(row).cuda()
    K.repack_row_to_tiled(buf, torch.empty(m * k // 2, dtype=torch.uint8, device="cuda"), m, k)
    torch.cuda.synchronize()
    got = buf.cpu().numpy()
    assert np.array_equal(got[:m * k // 2], O.fp4_to_tiled(row, m, k))
    assert (got[m * k // 2:] == 0xA5).all()
