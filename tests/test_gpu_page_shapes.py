"""The per-page NVFP4 kernels at the edges of their launch shapes: the K at which a row takes 16, 32
or 64 lanes and one or several passes, rows that are no whole wave, more row groups than resident
waves, and unaligned f32 / f16 activations. Block-scaled sums are exact in f64: bit for bit the
oracle's. The scalar kernels sum K products in f32: error at most K 2^-24 of the sum of magnitudes."""
import sys

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SHAPES = [(32, 1), (512, 5), (2048, 130), (2080, 33), (4096, 7), (4128, 65), (8192, 3), (8224, 70),
          (20000, 4), (64, 8200), (2112, 4100), (4160, 2050)]


def _page(rng, m, k, mantissa):
    data = rng.integers(0, 256, m * k // 2, dtype=np.uint8)
    s = rng.integers(119, 124, (m, k // 32)) << 7
    if mantissa:
        s |= rng.integers(0, 128, (m, k // 32))
    s = s.astype(np.uint16)
    return data, s, torch.from_numpy(np.concatenate([data, s.view(np.uint8).ravel()])).cuda()


def _dev_at(a, shift):
    """`a` on the device, `shift` elements past an aligned address."""
    t = torch.zeros(a.size + shift + 8, dtype=torch.from_numpy(a[:1]).dtype, device="cuda")
    t[shift:shift + a.size] = torch.from_numpy(a).cuda()
    return t[shift:]


def _out(m, dtype=torch.float32):
    return torch.full((m + 16,), 7.5, dtype=dtype, device="cuda")


@pytest.mark.parametrize("k,m", SHAPES)
def test_block_scaled(k, m):
    from vib3_amd import _lib, kernels as K
    print(f"case: block-scaled pages k={k} m={m}", flush=True)
    sys.stdout.flush()
    rng = np.random.default_rng(k + m)
    x = (rng.standard_normal(k) * 2).astype(np.float32)
    x[:32] *= np.float32(1e-39) if k > 32 else np.float32(1)  # a group below the E8M0 range
    codes, sc = O.fp4_quantize_act(x)
    a, asc = torch.from_numpy(codes).cuda(), torch.from_numpy(sc).cuda()
    (ud, us, up), (gd, gs, gp) = (_page(rng, m, k, False) for _ in range(2))
    fd, fs, fp = _page(rng, m, k, True)
    st = torch.cuda.current_stream().cuda_stream
    one, two, full, tiled, seq, seq2 = (_out(m) for _ in range(6))
    K.gemv_mma_nvfp4_preq(a, asc, up, one, k, m)
    K.fused_swiglu_mma_nvfp4_preq(a, asc, up, gp, two, k, m)
    _lib.call("vib3_launch_gemv_scalar_nvfp4", a.data_ptr(), asc.data_ptr(), fp.data_ptr(),
              fp.data_ptr() + fd.size, full.data_ptr(), k, m, st)
    if k % 64 == 0 and m % 16 == 0:
        _lib.call("vib3_launch_gemv_mma_nvfp4_tiled", a.data_ptr(), asc.data_ptr(), up.data_ptr(),
                  up.data_ptr() + ud.size, tiled.data_ptr(), k, m, st)
    K.gemv_mma_nvfp4(_dev_at(x, k % 3), up, seq, k, m)
    K.fused_swiglu_mma_nvfp4(_dev_at(x, 0), up, gp, seq2, k, m)
    torch.cuda.synchronize()
    want = {"one": (one, O.nvfp4_page_matvec(codes, sc, ud, us, m, k, 0)),
            "two": (two, O.nvfp4_page_swiglu(codes, sc, ud, us, gd, gs, m, k, 0)),
            "full": (full, O.nvfp4_page_matvec(codes, sc, fd, fs, m, k, 0, True)),
            "seq": (seq, O.nvfp4_page_matvec(codes, sc, ud, us, m, k, 2)),
            "seq2": (seq2, O.nvfp4_page_swiglu(codes, sc, O.fp4_split_half(ud), us, O.fp4_split_half(gd), gs, m, k, 0))}
    if k % 64 == 0 and m % 16 == 0:
        want["tiled"] = (tiled, O.nvfp4_page_matvec(codes, sc, ud, us, m, k, 1))
    for name, (got, ref) in want.items():
        g = got.cpu().numpy()
        assert np.array_equal(g[:m], ref), name
        assert (g[m:] == 7.5).all(), name


@pytest.mark.parametrize("k,m", [s for s in SHAPES if s[0] <= 16384])
def test_scalar(k, m):
    from vib3_amd import _lib
    print(f"case: scalar pages k={k} m={m}", flush=True)
    rng = np.random.default_rng(k * 3 + m)
    x = rng.standard_normal(k).astype(np.float16)
    d, s, p = _page(rng, m, k, True)
    xf = x.astype(np.float32)
    xd, xh = _dev_at(xf, m % 2), _dev_at(x, k % 3)
    st = torch.cuda.current_stream().cuda_stream
    got32, got16 = _out(m), _out(m, torch.float16)
    bs = 64 if k % 64 == 0 else 32
    for name, xin, out in (("f32out", xd, got32), ("fp16in", xh, got16)):
        _lib.call("vib3_launch_partial_matmul_nvfp4_" + name, xin.data_ptr(), p.data_ptr(),
                  p.data_ptr() + d.size, out.data_ptr(), k, m, bs, st)
    torch.cuda.synchronize()
    nb = k // bs
    # the page's scale words are read as [m][K / bs]; the oracle takes one per 32
    s32 = np.repeat(s.ravel()[:m * nb].reshape(m, nb), bs // 32, axis=1)
    want = O.nvfp4_seq_matvec_f64(xf, d, s32, m, k)
    mags = O.nvfp4_seq_matvec_f64(np.abs(xf), d & 0x77, s32, m, k)  # sum of |x w s|
    g32, g16 = got32.cpu().numpy(), got16.cpu().numpy()
    assert np.all(np.abs(g32[:m] - want) <= k * 2.0 ** -24 * mags + 1e-30)
    assert np.all(np.abs(g16[:m].astype(np.float64) - want) <= np.abs(want) * 2.0 ** -11 + 2.0 ** -24 + k * 2.0 ** -23 * mags)
    assert (g32[m:] == 7.5).all() and (g16[m:] == 7.5).all()


# Both sides of the lines between the row kernel and the staged one (16-row workgroups): short rows, many
# rows of each lane count, pairs and tiled pages earlier than single row-major ones; rows that are no
# whole workgroup, a staged activation near the longest the f32-input form takes.
CHOICE = [(64, 64), (1024, 65), (1056, 64), (1056, 65), (1024, 16), (2048, 2560), (2048, 2576), (2560, 6144), (2560, 6161),
          (4096, 6160), (3072, 10241), (3072, 12288), (3072, 12304), (4160, 6144), (4160, 6160), (4160, 8208), (4128, 12289),
          (20032, 6160)]


@pytest.mark.parametrize("k,m", CHOICE)
def test_block_scaled_kernel_choice(k, m):
    test_block_scaled(k, m)
