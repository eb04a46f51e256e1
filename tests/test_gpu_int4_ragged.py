"""The unaligned INT4 page kernel at its edges: k from one chunk up, odd k, k one past a multiple of
32, the k at which a row takes 16 / 32 / 64 lanes and several passes, few and many rows, pages and
activations at odd addresses with NaNs around the activation (no column outside it may count)."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# k, m, group, scale dtype, activation dtype, byte shift of the pages, element shift of x
CASES = [
    (32, 3, 32, O.BF16, O.F32, 1, 1), (33, 1, 32, O.F16, O.F16, 0, 0), (63, 70, 32, O.BF16, O.BF16, 0, 3),
    (64, 2100, 64, O.F16, O.F32, 8, 0), (95, 17, 96, O.BF16, O.F16, 3, 1), (1000, 520, 32, O.BF16, O.F32, 0, 0),
    (1364, 333, 128, O.F16, O.F16, 0, 1), (2047, 4097, 32, O.BF16, O.F16, 0, 0), (2049, 1030, 64, O.F16, O.F32, 2, 0),
    (4095, 2, 32, O.BF16, O.BF16, 0, 1), (4129, 1025, 32, O.BF16, O.F32, 0, 2), (8191, 9, 128, O.F16, O.F16, 1, 0),
    (8193, 40, 32, O.BF16, O.F32, 0, 0), (14337, 5, 96, O.F16, O.BF16, 5, 1), (7168, 600, 32, O.BF16, O.BF16, 4, 0),
]


def _at(a, shift, fill):
    """Device copy of `a`, `shift` elements past a 256-byte boundary, `fill` all around it."""
    t = torch.from_numpy(np.full(a.size + shift + 64, fill, dtype=a.dtype)).cuda()
    t[shift:shift + a.size] = torch.from_numpy(a).cuda()
    return t[shift:]


@pytest.mark.parametrize("k,m,g,sdt,adt,pshift,xshift", CASES)
def test_ragged_pages(k, m, g, sdt, adt, pshift, xshift):
    from vib3_amd import _lib
    print(f"case: ragged k={k} m={m} g={g} sdt={sdt} adt={adt} shifts={pshift},{xshift}", flush=True)
    bits = O.synth_normal_array(7, 100 + k, 0, k, 1.0, adt)
    xh = bits if adt == O.F32 else O.to_f32(bits, adt)
    nan = {O.F32: np.float32(np.nan), O.F16: 0x7E00, O.BF16: 0x7FC0}[adt]
    x = _at(bits, xshift, nan)
    if xshift:
        x0 = x.storage_offset()
        x._base[:x0] = float("nan") if adt == O.F32 else torch.tensor(int(nan), dtype=torch.int32).to(x.dtype)
    pages = [O.synth_int4_page(0x5EED0000, s + k, k, g, sdt, 0.02, 0, m) for s in (2000, 3000)]
    up, gate = (_at(p, pshift, 0xFF) for p in pages)
    st = torch.cuda.current_stream().cuda_stream
    out = torch.full((m + 8,), 7.5, dtype=torch.float32, device="cuda")
    out16 = torch.full((m + 8,), 7.5, dtype=torch.float16, device="cuda")
    two = out.clone()
    for o, dt in ((out, _lib.DT_F32), (out16, _lib.DT_F16)):
        _lib.call("vib3_launch_partial_matmul_int4_ex", x.data_ptr(), adt, up.data_ptr(), o.data_ptr(), dt, k, m, g,
                  sdt, st)
    _lib.call("vib3_launch_partial_swiglu_int4_ex", x.data_ptr(), adt, up.data_ptr(), gate.data_ptr(),
              two.data_ptr(), _lib.DT_F32, k, m, g, sdt, st)
    torch.cuda.synchronize()
    ref = O.matmul_int4_acc(xh, pages[0], k, m, g, sdt).astype(np.float64)
    ref2 = O.swiglu_int4_acc(xh, pages[0], pages[1], k, m, g, sdt).astype(np.float64)
    o, t = out.cpu().numpy(), two.cpu().numpy()
    # f32 sums of k <= 16384 terms in another order: rel-L2 5e-5, as for the aligned kernels
    assert np.linalg.norm(o[:m] - ref) <= 5e-5 * np.linalg.norm(ref)
    assert np.linalg.norm(t[:m] - ref2) <= 5e-5 * np.linalg.norm(ref2)
    assert np.array_equal(out16.cpu().numpy()[:m], o[:m].astype(np.float16))
    assert (o[m:] == 7.5).all() and (t[m:] == 7.5).all()
