"""INT4 group sizes that are no multiple of 32, where the chunk kernels' one scale per 32 columns does
not hold: aligned pages (which took the chunk kernels by shape alone), unaligned ones and one group per
row, against the oracle; the fused layer, which has no other kernel, refuses them."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O

# k, m, group: below a chunk, between chunks, one group per row with and without a round size, k > 8192
CASES = [(1024, 70, 16), (96, 5, 48), (256, 33, 100), (96, 40, 96), (96, 40, 100), (8224, 9, 48), (1000, 21, 24)]


@pytest.mark.gpu
@pytest.mark.parametrize("k,m,g", CASES)
@pytest.mark.parametrize("adt", [O.F32, O.F16])
def test_group_sizes(k, m, g, adt):
    import torch
    from vib3_amd import _lib
    print(f"case: groups k={k} m={m} g={g} adt={adt}", flush=True)
    bits = O.synth_normal_array(7, 400 + k, 0, k, 1.0, adt)
    xh = bits if adt == O.F32 else O.to_f32(bits, adt)
    pages = [O.synth_int4_page(0x5EED0000, s + k, k, g, O.BF16, 0.02, 0, m) for s in (5000, 6000)]
    x = torch.from_numpy(bits if adt == O.F32 else bits.view(np.int16)).cuda()
    up, gate = (torch.from_numpy(p).cuda() for p in pages)
    out = torch.full((m + 8,), 7.5, dtype=torch.float32, device="cuda")
    two = out.clone()
    st = torch.cuda.current_stream().cuda_stream
    _lib.call("vib3_launch_partial_matmul_int4_ex", x.data_ptr(), adt, up.data_ptr(), out.data_ptr(), _lib.DT_F32, k,
              m, g, O.BF16, st)
    _lib.call("vib3_launch_partial_swiglu_int4_ex", x.data_ptr(), adt, up.data_ptr(), gate.data_ptr(),
              two.data_ptr(), _lib.DT_F32, k, m, g, O.BF16, st)
    torch.cuda.synchronize()
    o, t = out.cpu().numpy(), two.cpu().numpy()
    ref = O.matmul_int4_acc(xh, pages[0], k, m, g, O.BF16).astype(np.float64)
    ref2 = O.swiglu_int4_acc(xh, pages[0], pages[1], k, m, g, O.BF16).astype(np.float64)
    # f32 sums in another order: rel-L2 5e-5, as for the other INT4 kernels
    assert np.linalg.norm(o[:m] - ref) <= 5e-5 * np.linalg.norm(ref)
    assert np.linalg.norm(t[:m] - ref2) <= 5e-5 * np.linalg.norm(ref2)
    assert (o[m:] == 7.5).all() and (t[m:] == 7.5).all()


@pytest.mark.parametrize("g", [16, 48, 100, 1000])
def test_layer_refuses_groups_inside_a_chunk(g):
    """Refused by the argument checks, before anything is launched (no pointer here is real)."""
    from vib3_amd import _lib
    d = _lib.MoeInt4Layer()
    d.x, d.x_dtype, d.hidden, d.inter, d.group_size, d.scale_dtype = 1 << 20, _lib.DT_F16, 1024, 512, g, _lib.DT_F16
    d.num_experts, d.top_k, d.max_pages = 4, 2, 1
    d.rows_per_page[0], d.rows_per_page[1], d.rows_per_page[2] = 512, 512, 1024
    d.page_table, d.out, d.workspace = 1 << 21, 1 << 22, 1 << 23
    d.in_ids, d.in_weights = 1 << 24, 1 << 24
    lib = _lib.load()
    d.workspace_bytes = lib.vib3_moe_int4_workspace_bytes(C.byref(d))
    assert lib.vib3_launch_moe_int4_layer(C.byref(d), None) == -1
    assert lib.vib3_launch_moe_int4_layer_stage(C.byref(d), 2, None) == -1
