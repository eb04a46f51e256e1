"""One INT4 page with k > 8192 and f16 activations: the staged-activation kernel (one chunk past four
per lane, no multiple of a pass, the longest k its LDS holds, one to four rows per wave, few rows), and
the shapes just outside it (scales not behind the rows, k past its LDS, row counts at which the split
kernel is faster) that keep the split kernel."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("k,m,g,sdt,apart", [
    # both sides of the lines between the two kernels, and of those between 1, 2 and 4 rows per wave
    (8224, 2049, 32, O.BF16, False), (8224, 4097, 32, O.F16, False), (8224, 8193, 32, O.BF16, False),
    (12288, 14337, 128, O.F16, False), (14336, 7169, 128, O.F16, False), (18432, 4, 32, O.BF16, False),
    (18432, 5, 32, O.BF16, False), (20480, 4100, 128, O.BF16, False), (24576, 4097, 128, O.F16, False),
    (24576, 6145, 128, O.F16, False), (28672, 2049, 128, O.BF16, False),
    (8224, 1, 32, O.BF16, False), (8224, 523, 64, O.F16, False), (9216, 3073, 32, O.BF16, False),
    (14336, 6149, 128, O.F16, False), (30816, 5, 32, O.BF16, False), (30848, 5, 32, O.BF16, False),
    (8224, 37, 32, O.F16, True)])
def test_long_k(k, m, g, sdt, apart):
    from vib3_amd import _lib
    print(f"case: long k={k} m={m} g={g} sdt={sdt} apart={apart}", flush=True)
    x = O.synth_normal_array(7, 300 + k, 0, k, 1.0, O.F16)
    page = O.synth_int4_page(0x5EED0000, 4000 + k, k, g, sdt, 0.02, 0, m)
    xd = O.to_f32(x, O.F16).astype(np.float64)
    b = page[:m * k // 2].reshape(m, k // 2)
    q = np.stack([b & 15, b >> 4], 2).reshape(m, k).astype(np.float64) - 8
    s = O.to_f32(page[m * k // 2:].view(np.uint16), sdt).astype(np.float64).reshape(m, -(-k // g)).repeat(g, 1)[:, :k]
    ref = (q * s) @ xd
    # f32: the roundings a term passes, in either kernel: 31 in its chunk's offset term (32 activations
    # added one after another; the codes' side has 16 two-term dot products over two sums, 17), 1 where the
    # offset is subtracted, 16 multiply-adds of its lane's chunks (1024 chunks over 64 lanes), 6 of the sum
    # over lanes, 3 of the sum over up to four waves: 57, taken as 60. Each is at most 2^-24 of a partial
    # sum no larger than the sum of |x| (|q - 8| + 8) s.
    bound = 60 * 2.0 ** -24 * (((np.abs(q) + 8) * s) @ np.abs(xd))
    dx, dp = torch.from_numpy(x.view(np.int16)).cuda(), torch.from_numpy(page).cuda()
    st = torch.cuda.current_stream().cuda_stream
    out = torch.full((m + 8,), 7.5, dtype=torch.float32, device="cuda")
    out16 = torch.full((m + 8,), 7.5, dtype=torch.float16, device="cuda")
    if apart:  # f16 scales in a buffer of their own: the reference's launcher, f16 out only
        sc = dp[m * k // 2:].clone()
        _lib.call("vib3_launch_partial_matmul_int4", dx.data_ptr(), dp.data_ptr(), sc.data_ptr(), out16.data_ptr(),
                  k, m, g, st)
    else:
        for o, dt in ((out, _lib.DT_F32), (out16, _lib.DT_F16)):
            _lib.call("vib3_launch_partial_matmul_int4_ex", dx.data_ptr(), O.F16, dp.data_ptr(), o.data_ptr(), dt, k,
                      m, g, sdt, st)
    torch.cuda.synchronize()
    o, o16 = out.cpu().numpy(), out16.cpu().numpy()
    assert (o[m:] == 7.5).all() and (o16[m:] == 7.5).all()
    if not apart:
        assert np.all(np.abs(o[:m] - ref) <= bound)
        assert np.array_equal(o16[:m], o[:m].astype(np.float16))
    assert np.all(np.abs(o16[:m].astype(np.float64) - ref) <= bound + np.abs(ref) * 2.0 ** -11 + 2.0 ** -24)
