"""The unaligned INT4 page kernels at their edges: k from one chunk up, odd k, k one past a multiple of
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


# Both sides of the lines between this kernel and the per-column one: rows of two and three chunks, pairs
# of four and five, and pairs of many rows.
CHOICE = [(64, 300, 32, O.BF16, O.F16, 8, 1), (65, 300, 32, O.BF16, O.F32, 0, 0), (96, 9, 64, O.F16, O.BF16, 1, 0),
          (128, 130, 32, O.BF16, O.F16, 2, 0), (129, 130, 32, O.BF16, O.F16, 0, 1), (100, 8191, 32, O.BF16, O.F32, 0, 0),
          (100, 8192, 32, O.BF16, O.F32, 0, 0), (127, 8193, 64, O.F16, O.F16, 0, 0)]


@pytest.mark.parametrize("k,m,g,sdt,adt,pshift,xshift", CHOICE)
def test_ragged_kernel_choice(k, m, g, sdt, adt, pshift, xshift):
    test_ragged_pages(k, m, g, sdt, adt, pshift, xshift)


def _page(codes, scales):
    """One INT4 page from codes [m][k] (0..15) and scales [m][groups] as bf16 bits."""
    m, k = codes.shape
    c = np.zeros((m, 2 * ((k + 1) // 2)), dtype=np.uint8)
    c[:, :k] = codes
    return np.concatenate([(c[:, ::2] | (c[:, 1::2] << 4)).ravel(), scales.astype(np.uint16).view(np.uint8).ravel()])


@pytest.mark.parametrize("k,m", [(1000, 8), (2049, 8), (8193, 8), (1000, 8 * 1024 + 5)])
def test_ragged_large_and_infinite_values(k, m):
    """Terms x ((q - 8) scale) far below the f32 limit whose x (q - 8) is above it sum to what the terms
    do; an infinite activation comes through as in the term-by-term sum; scales that are no positive
    number read as 1/8, also the last group's, which lanes without a chunk of their own load too."""
    from vib3_amd import _lib
    print(f"case: ragged large values k={k} m={m}", flush=True)
    g = 32
    rng = np.random.default_rng(k)
    ng = -(-k // g)
    codes = rng.integers(0, 16, (m, k))
    scales = np.full((m, ng), 0x3080)  # bf16 2^-30
    scales[0, ng - 1], scales[1, 5], scales[2, ng - 2] = 0x7F80, 0x7FC0, 0xFF80  # inf, NaN, -inf
    x = rng.standard_normal(k).astype(np.float32)
    big, bad = x.copy(), x.copy()
    big[40:72] = 2.0e38            # x (q - 8) passes 2^128, every term stays below 2^125
    codes[4, 40:72] = 15
    bad[k - 1] = np.inf
    codes[:, k - 1] = np.where(np.arange(m) == 3, 8, 9)  # row 3: inf * 0
    s = (scales.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    s = np.where(np.isfinite(s) & (s > 0), s, 0.125)
    page = torch.from_numpy(_page(codes, scales)).cuda()
    for xv in (x, big, bad):
        with np.errstate(invalid="ignore"):
            terms = xv.astype(np.float64) * ((codes - 8) * s.repeat(g, 1)[:, :k])
            ref = terms.sum(1)
            # k f32 additions in any order and one product per term: (k + 2) roundings
            bound = (k + 2) * 2.0 ** -24 * np.abs(terms).sum(1)
        xd = torch.from_numpy(xv).cuda()
        out = torch.empty(m, dtype=torch.float32, device="cuda")
        two = torch.empty(m, dtype=torch.float32, device="cuda")
        st = torch.cuda.current_stream().cuda_stream
        _lib.call("vib3_launch_partial_matmul_int4_ex", xd.data_ptr(), O.F32, page.data_ptr(), out.data_ptr(),
                  _lib.DT_F32, k, m, g, O.BF16, st)
        _lib.call("vib3_launch_partial_swiglu_int4_ex", xd.data_ptr(), O.F32, page.data_ptr(), page.data_ptr(),
                  two.data_ptr(), _lib.DT_F32, k, m, g, O.BF16, st)
        torch.cuda.synchronize()
        o, t = out.cpu().numpy(), two.cpu().numpy()
        fin = np.isfinite(ref)
        assert np.array_equal(np.isnan(o), np.isnan(ref)) and np.array_equal(np.isinf(o), np.isinf(ref)), (o, ref)
        assert (np.abs(o[fin] - ref[fin]) <= bound[fin]).all(), (o, ref)
        with np.errstate(invalid="ignore", over="ignore"):
            sw = (o / (np.float32(1) + np.exp(-o))) * o  # silu(gate) * up of the same sums
        assert np.array_equal(np.isfinite(t), np.isfinite(sw)), (t, sw)
