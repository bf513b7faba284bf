"""GPU parity of the N-d linear sampler (forward, grad-data, grad-coord) against the CPU
oracle.  fp32: forward 1e-5 against the fp32 oracle, gradients 1e-4 against the fp64 oracle;
fp64 1e-11; fp16 / bf16 1e-2 against the fp32 oracle on the rounded inputs."""
import numpy as np
import pytest
import torch

from _cases import rel_err
from oracle import dk_oracle as orc

pytestmark = pytest.mark.gpu


def _inputs(shape, C, B, seed, dtype, lo=-1.5, extra=1.5):
    g = torch.Generator().manual_seed(seed)
    data = torch.randn(C, *shape, generator=g)
    hi = torch.tensor(shape, dtype=torch.float32)
    coord = torch.rand(B, len(shape), generator=g) * (hi + extra - lo) + lo  # spills outside on both sides
    gout = torch.randn(B, C, generator=g)
    return data.to(dtype), coord.to(dtype), gout.to(dtype)


def _run(data, coord, gout):
    from deformable_kernels.ops.deform_kernel.functions import nd_linear_sample
    dev = torch.device("cuda:0")
    dg, cg = data.to(dev).requires_grad_(), coord.to(dev).requires_grad_()
    out = nd_linear_sample(dg, cg)
    out.backward(gout.to(dev))
    torch.cuda.synchronize()
    return out.detach().cpu(), dg.grad.cpu(), cg.grad.cpu()


def _oracle(data, coord, gout, np_dtype):
    a = [t.to(torch.float64).numpy().astype(np_dtype) for t in (data, coord, gout)]
    out = orc.nd_linear_sample_forward(a[0], a[1])
    gd, gc = orc.nd_linear_sample_backward(a[2], a[0], a[1])
    return out, gd, gc


@pytest.mark.parametrize("shape,C,B", [((9,), 5, 70), ((5, 5), 256, 1152), ((4, 5, 6), 7, 333),
                                       ((3, 4, 2, 5), 3, 200), ((2, 2), 1, 1),
                                       ((9,), 40, 3000), ((6, 7, 5), 100, 1001), ((5, 4), 16, 4097)])
def test_fp32_matches_oracle(shape, C, B):
    data, coord, gout = _inputs(shape, C, B, seed=41, dtype=torch.float32)
    got = _run(data, coord, gout)
    o32, o64 = _oracle(data, coord, gout, np.float32), _oracle(data, coord, gout, np.float64)
    assert got[0].shape == (B, C)
    assert rel_err(got[0], o32[0]) < 1e-5
    assert rel_err(got[1], o64[1]) < 1e-4
    assert rel_err(got[2], o64[2]) < 1e-4


@pytest.mark.parametrize("shape,C,B,lo,hi", [
    ((8, 8, 8), 64, 65536 + 37, -1.5, 9.5),    # many points per cell: the sorted-by-cell kernels; ragged last wave
    ((16, 12), 80, 70001, -1.5, 17.0),         # two channel passes (64 + 16)
    ((40,), 16, 66000, -2.0, 42.0),            # one dimension
    ((8, 8, 8), 32, 65536, -1.0, 1.0),         # config 5's coordinate range: every point in the 8 corner cells
    ((6, 5, 4), 64, 65536, 2.2, 2.9),          # every point in one cell
    ((10, 9), 128, 66000, -1.5, 10.5),         # two dimensions, two 64-channel blocks of the matrix-core kernels
    ((50,), 64, 66000, -2.0, 52.0),            # one dimension on the matrix-core kernels
    ((5, 6, 7), 192, 65536, -1.5, 7.5),        # three 64-channel blocks
])
def test_many_points_per_cell_match_oracle(shape, C, B, lo, hi):
    g = torch.Generator().manual_seed(45)
    data = torch.randn(C, *shape, generator=g)
    coord = torch.rand(B, len(shape), generator=g) * (hi - lo) + lo
    gout = torch.randn(B, C, generator=g)
    got = _run(data, coord, gout)
    o32, o64 = _oracle(data, coord, gout, np.float32), _oracle(data, coord, gout, np.float64)
    assert rel_err(got[0], o32[0]) < 1e-5
    assert rel_err(got[1], o64[1]) < 1e-4
    assert rel_err(got[2], o64[2]) < 1e-4


def test_many_points_on_grid_nodes_and_half_way_between():
    # fractional positions of exactly 0 and 0.5: a corner with interpolation weight 0 still
    # enters the coordinate gradient
    g = torch.Generator().manual_seed(47)
    data = torch.randn(32, 7, 6, 5, generator=g)
    hi = torch.tensor([7.0, 6.0, 5.0])
    coord = torch.round((torch.rand(65536, 3, generator=g) * (hi + 2.0) - 1.0) * 2.0) / 2.0
    gout = torch.randn(65536, 32, generator=g)
    got = _run(data, coord, gout)
    o32, o64 = _oracle(data, coord, gout, np.float32), _oracle(data, coord, gout, np.float64)
    assert rel_err(got[0], o32[0]) < 1e-5
    assert rel_err(got[1], o64[1]) < 1e-4
    assert rel_err(got[2], o64[2]) < 1e-4


def test_sorted_and_unsorted_kernels_agree(switch_off):
    g = torch.Generator().manual_seed(46)
    data = torch.randn(64, 8, 8, 8, generator=g)
    coord = torch.rand(70000, 3, generator=g) * 10.0 - 1.0
    gout = torch.randn(70000, 64, generator=g)
    a = _run(data, coord, gout)
    switch_off("DK_NO_ND_BINS")
    b = _run(data, coord, gout)
    assert rel_err(a[0], b[0]) < 1e-6  # the same eight products per point and channel, summed in another order
    assert rel_err(a[1], b[1]) < 1e-5
    assert rel_err(a[2], b[2]) < 1e-5


def test_sorted_kernels_with_and_without_the_matrix_cores_agree(switch_off):
    """64 channels in fp32 take the matrix-core kernels; switched off, the VALU kernels serve the same call."""
    g = torch.Generator().manual_seed(47)
    data = torch.randn(64, 7, 9, 8, generator=g)
    coord = torch.rand(66000, 3, generator=g) * 11.0 - 1.5
    gout = torch.randn(66000, 64, generator=g)
    a = _run(data, coord, gout)
    switch_off("DK_NO_ND_MFMA")
    b = _run(data, coord, gout)
    want = _oracle(data, coord, gout, np.float64)
    for x, y, w in zip(a, b, want):
        assert rel_err(x, y) < 1e-5
        assert rel_err(y, w) < 1e-4


@pytest.mark.parametrize("dtype,C,B", [(torch.float32, 256, 1152), (torch.float16, 64, 4096), (torch.bfloat16, 100, 700)])
def test_channel_last_kernels_on_few_points_over_a_tiny_volume(dtype, C, B, switch_off):
    """Few points on a volume of at most 64 cells take the direct kernels and the one-launch grad
    data; with that path switched off the channel-last kernels serve the same call."""
    data, coord, gout = _inputs((5, 5), C, B, seed=44, dtype=dtype)
    small = _run(data, coord, gout)
    switch_off("DK_NO_ND_SMALL")
    general = _run(data, coord, gout)
    want = _oracle(data, coord, gout, np.float64)
    tol = (1e-5, 1e-4, 1e-4) if dtype == torch.float32 else (1e-2, 1e-2, 1e-2)
    for a, b, w, t in zip(small, general, want, tol):
        assert rel_err(a.float(), w) < t
        assert rel_err(b.float(), w) < t


def test_fp64_matches_oracle():
    data, coord, gout = _inputs((4, 5, 6), 9, 257, seed=42, dtype=torch.float64)
    got = _run(data, coord, gout)
    want = _oracle(data, coord, gout, np.float64)
    for g, w in zip(got, want):
        assert rel_err(g, w) < 1e-11


@pytest.mark.parametrize("points", [300, 4096, 65536])   # direct path / channel-last path / sorted by cell
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_half_precisions_match_fp32_oracle(dtype, points):
    data, coord, gout = _inputs((5, 5), 64, points, seed=43, dtype=dtype)
    got = _run(data, coord, gout)
    want = _oracle(data, coord, gout, np.float32)
    for g, w in zip(got, want):
        assert g.dtype == dtype
        assert rel_err(g.float(), w) < 1e-2


def test_zero_rule_and_fade_bands_on_gpu():
    data = torch.ones(1, 4, 4)
    pts = torch.tensor([[-1.0, 1.0], [1.0, -1.0], [4.0, 1.0], [1.0, 4.0], [-0.5, 1.0], [3.5, 3.5], [3.0, 3.0]])
    out, _, gc = _run(data, pts, torch.ones(7, 1))
    assert out[:4, 0].tolist() == [0, 0, 0, 0]
    assert torch.allclose(out[4:, 0], torch.tensor([0.5, 0.25, 1.0]))
    assert torch.count_nonzero(gc[:4]).item() == 0


def test_trilinear_volume_slice_of_config5():
    """Config 5's standalone case at reduced point count: data [64, 32, 32, 32], coordinates
    uniform in [-1, 1]^3 as written there (half the points in the fade band) and uniform over
    the whole volume."""
    g = torch.Generator().manual_seed(44)
    data = torch.randn(64, 32, 32, 32, generator=g)
    for lo, hi in ((-1.0, 1.0), (-1.0, 32.0)):
        coord = torch.rand(4096, 3, generator=g) * (hi - lo) + lo
        gout = torch.randn(4096, 64, generator=g)
        got = _run(data, coord, gout)
        o32, o64 = _oracle(data, coord, gout, np.float32), _oracle(data, coord, gout, np.float64)
        assert rel_err(got[0], o32[0]) < 1e-5
        assert rel_err(got[1], o64[1]) < 1e-4
        assert rel_err(got[2], o64[2]) < 1e-4


@pytest.mark.parametrize("shape,C,B", [
    ((6, 5, 4), 64, 65536),      # a cell holds several waves' points
    ((12, 11, 10), 128, 65537),  # two channel blocks: the coordinates' gradient is added up over them; one point in the last wave
    ((33, 40), 64, 65599),       # two dimensions, runs of about 45 points
    ((900,), 64, 65600),         # one dimension
])
def test_both_gradients_of_sorted_points_equal_those_formed_alone(shape, C, B):
    """One kernel forms both from one read of the output gradient; with a single input to differentiate each has its own.  The
    same products in another order: a few units of 2^-24 of the sums' size."""
    from deformable_kernels.ops.deform_kernel.functions import nd_linear_sample
    data, coord, gout = _inputs(shape, C, B, seed=48, dtype=torch.float32)
    outside = (coord <= -1).any(1) | (coord >= torch.tensor(shape, dtype=torch.float32)).any(1)
    gout[outside.nonzero()[0, 0]] = float("inf")  # an output gradient that a point outside the grid multiplies with nothing
    dg, cg = data.cuda().requires_grad_(), coord.cuda().requires_grad_()
    out = nd_linear_sample(dg, cg)
    both = torch.autograd.grad(out, [dg, cg], gout.cuda(), retain_graph=True)
    alone = torch.autograd.grad(out, [cg], gout.cuda(), retain_graph=True)[0]
    gout[outside] = 0.0
    want = _oracle(data, coord, gout, np.float64)
    assert rel_err(both[0].cpu(), want[1]) < 1e-5 and rel_err(both[1].cpu(), want[2]) < 1e-5
    assert rel_err(both[1].cpu(), alone.double().cpu().numpy()) < 1e-6


@pytest.mark.parametrize("B", [1 << 20, (1 << 20) + 1])
def test_sort_on_either_side_of_the_most_tiles_that_the_scatter_sums_itself(B):
    """18 key bits, 512 or 513 workgroups: 64 tiles of the digit table, whose sums the scatter adds up itself, and 65, which have a
    kernel for that.  An output is two products and a sum: 3 * 2^-24 of its operands' size; a gradient sums some ten."""
    S, C = 200000, 16
    data, coord, gout = _inputs((S,), C, B, seed=49, dtype=torch.float32, lo=0.0, extra=-2.0)
    data, coord, gout = (t.cuda() for t in (data, coord, gout))
    dg = data.requires_grad_()
    from deformable_kernels.ops.deform_kernel.functions import nd_linear_sample
    out = nd_linear_sample(dg, coord)
    grad = torch.autograd.grad(out, dg, gout)[0]
    low = coord[:, 0].floor().long()
    frac = (coord[:, 0] - low).double()
    rows = data.detach().double().t().contiguous()
    want = rows[low] * (1 - frac)[:, None] + rows[low + 1] * frac[:, None]
    assert float((out.detach() - want).abs().max()) < 3 * 2.0 ** -24 * 2 * float(data.detach().abs().max())
    want = torch.zeros_like(rows).index_add_(0, low, gout.double() * (1 - frac)[:, None])
    want.index_add_(0, low + 1, gout.double() * frac[:, None])
    assert rel_err(grad.cpu(), want.t().cpu().numpy()) < 1e-5


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.float64])
def test_both_gradients_of_no_points_through_the_c_call(dtype):
    """As dk_nd_linear_sample_backward_data: zeros in in_grad, and nothing else is looked at."""
    from deformable_kernels.ops.deform_kernel import _lib
    L, P = _lib.lib(), _lib.ptr
    gdata = torch.full((64, 6, 5, 4), float("nan"), device="cuda:0", dtype=dtype)
    desc = _lib.NdDesc()
    desc.batch, desc.channel, desc.dims = 0, 64, 3
    desc.dtype = {torch.float32: 0, torch.float16: 1, torch.float64: 3}[dtype]
    for d, n in enumerate((6, 5, 4)):
        desc.shape[d] = n
    ws, n = _lib.workspace(L.dk_nd_linear_sample_backward_workspace(desc), gdata.device)
    _lib.check(L.dk_nd_linear_sample_backward(desc, None, None, None, None, P(gdata), None, P(ws), n, _lib.stream_ptr(gdata)), "backward")
    assert bool((gdata == 0).all())


@pytest.mark.parametrize("shape,C,B,lo,hi", [
    ((20, 31), 14, 9001, -1.5, 32.0),        # narrow rows, a lane group partly idle; the sums in LDS
    ((90,), 1, 70000, -1.0, 90.0),           # one channel, a lane per point
    ((13, 9, 8), 3, 30011, -1.5, 13.5),
    ((6, 12), 11, 20000, 2.0, 2.9),          # every point in one cell
    ((70, 78), 15, 30000, -1.0, 78.0),       # five slices of channels
    ((40, 40, 40), 2, 70000, -1.0, 40.0),    # one channel in four ranges of cells, two slices
    ((28, 28, 24), 4, 70000, -1.0, 28.0),    # 18816 cells: one channel per workgroup, one range
    ((80, 80, 80), 5, 20000, -1.0, 80.0),    # fewer additions than the sums in LDS want: float atomics
    ((40, 30), 17, 30000, -1.5, 41.0),       # 32 lanes per point
    ((40, 30), 32, 20000, -1.5, 41.0),
    ((40, 30), 33, 20000, -1.5, 41.0),       # a wave per point forward, the sums in LDS
    ((8, 8, 8), 20, 66000, -1.5, 9.0),       # two slices: not sorted
    ((7, 7), 16, 4097, -1.5, 8.0),           # a tiny volume, one point more than the few-points kernels take
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_narrow_rows_and_sums_in_lds(shape, C, B, lo, hi, dtype, switch_off):
    """Against float64, and against the kernels that take the calls without these."""
    g = torch.Generator().manual_seed(50)
    data = torch.randn(C, *shape, generator=g).to(dtype)
    coord = (torch.rand(B, len(shape), generator=g) * (hi - lo) + lo).to(dtype)
    gout = torch.randn(B, C, generator=g).to(dtype)
    got = _run(data, coord, gout)
    switch_off("DK_NO_ND_ROWS")
    general = _run(data, coord, gout)
    want = _oracle(data, coord, gout, np.float64)
    tol = (1e-5, 1e-5, 1e-5) if dtype == torch.float32 else (1e-3, 1e-3, 1e-3)  # 16-bit: the results' rounding, 2^-11
    for a, b, w, t in zip(got, general, want, tol):
        assert rel_err(a.float(), w) < t and rel_err(a.float(), b.double().numpy()) < t


def test_non_finite_output_gradient_stays_with_its_point_and_channel():
    """Sums in LDS: what is not finite reaches the corners of its point in its channel, and nothing else; a point outside the grid
    adds nothing."""
    data, coord, gout = _inputs((20, 31), 6, 20000, seed=51, dtype=torch.float32)
    coord[0], coord[1] = torch.tensor([3.25, 4.5]), torch.tensor([-1.0, 4.0])
    gout[0, 2], gout[1, 3] = float("inf"), float("nan")
    got = _run(data, coord, gout)[1]
    bad = ~torch.isfinite(got)
    assert bad[2, 3:5, 4:6].all() and int(bad.sum()) == 4


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_volume_of_more_cells_than_32_times_65535(dtype):
    """Both transposes: their tiles along the cells outnumber the second dimension of a grid."""
    data, coord, gout = _inputs((130, 130, 130), 16, 4500, seed=52, dtype=dtype)
    for a, w in zip(_run(data, coord, gout), _oracle(data, coord, gout, np.float64)):
        assert rel_err(a.float(), w) < (1e-5 if dtype == torch.float32 else 8e-3)  # bfloat16: the results' rounding, 2^-8


def _workspaces(dtype, C, shape, B):
    import ctypes
    from deformable_kernels.ops.deform_kernel import _lib
    L = _lib.lib()
    desc = _lib.NdDesc(B, C, len(shape), (ctypes.c_int32 * 8)(*shape, *([1] * (8 - len(shape)))), dtype)
    return [getattr(L, f"dk_nd_linear_sample_{k}_workspace")(ctypes.byref(desc)) for k in ("forward", "backward_data", "backward_coord")]


@pytest.mark.parametrize("shape,C,B,lo,hi,route", [
    ((20, 31), 14, 36000, -1.5, 32.0, "gradients"),   # 2.0 * 10^6 corners times channels of 620 cells
    ((20, 31), 14, 45000, -1.5, 32.0, "copied"),      # 2.52 * 10^6: the forward as well
    ((2000, 1500), 3, 30000, -1.0, 1500.0, "planar"),  # a volume that the points hardly read
    ((80, 80, 80), 5, 30000, -1.0, 80.0, "gradients"),  # 1.2 * 10^6, 512000 cells; float atomics
    ((80, 80, 80), 5, 62500, -1.0, 80.0, "copied"),   # 2.5 * 10^6
    ((80, 80, 80), 5, 20000, -1.0, 80.0, "planar"),   # 0.8 * 10^6
    ((100, 100, 100), 2, 90000, -1.0, 100.0, "planar"),   # 1.44 * 10^6 of 10^6 cells
    ((100, 100, 100), 2, 94000, -1.0, 100.0, "gradients"),   # 1.504 * 10^6
    ((100, 100, 100), 2, 157000, -1.0, 100.0, "copied"),   # 2.512 * 10^6, 2.5 per cell
    ((64, 64, 64), 1, 65536, -1.0, 64.0, "in place"),  # one channel: no sums in LDS
    ((64, 64, 64), 1, 140000, -1.0, 64.0, "in place"),  # ... with them
    ((1, 70000), 1, 66000, -1.0, 70000.0, "in place"),
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_few_channels_of_volumes_larger_than_what_is_read(shape, C, B, lo, hi, route, dtype):
    from deformable_kernels.ops.deform_kernel import _lib
    ws = _workspaces(_lib.DK_F32 if dtype == torch.float32 else _lib.DK_F16, C, shape, B)
    assert (ws[2] > 0) == (route in ("copied", "gradients")) and (ws[0] > 0) == (route == "copied")
    if dtype == torch.float16 and max(shape) > 2000:
        pytest.skip("coordinates that float16 does not hold")
    g = torch.Generator().manual_seed(53)
    data = torch.randn(C, *shape, generator=g).to(dtype)
    coord = (torch.rand(B, len(shape), generator=g) * (hi - lo) + lo).to(dtype)
    gout = torch.randn(B, C, generator=g).to(dtype)
    for a, w in zip(_run(data, coord, gout), _oracle(data, coord, gout, np.float64)):
        assert rel_err(a.float(), w) < (1e-5 if dtype == torch.float32 else 1e-3)  # 16-bit: the results' rounding, 2^-11


def test_non_finite_output_gradient_stays_with_its_point_and_channel_in_sums_of_many_points():
    data, coord, gout = _inputs((20, 31), 6, 40000, seed=51, dtype=torch.float32)
    coord[0], coord[1] = torch.tensor([3.25, 4.5]), torch.tensor([-1.0, 4.0])
    gout[0, 2], gout[1, 3] = float("inf"), float("nan")
    got = _run(data, coord, gout)[1]
    bad = ~torch.isfinite(got)
    assert bad[2, 3:5, 4:6].all() and int(bad.sum()) == 4


def test_more_points_than_threads_of_a_launch():
    """One channel, 2^32 + 77 points: the rows' kernels walk over them.  Every 2^16 points repeat, so the results do."""
    from deformable_kernels.ops.deform_kernel.functions import nd_linear_sample
    if torch.cuda.mem_get_info()[0] < 64 << 30:
        pytest.skip("needs 35 GB of GPU memory")
    n, period, dev = (1 << 32) + 77, 1 << 16, torch.device("cuda:0")
    g = torch.Generator().manual_seed(54)
    data, one = torch.randn(1, 90, generator=g).half().to(dev), (torch.rand(period, 1, generator=g) * 91 - 1).half().to(dev)
    gone = torch.randn(period, 1, generator=g).half().to(dev)

    def spread(t):
        full = torch.empty(n, 1, dtype=t.dtype, device=dev)
        full[:1 << 32].view(-1, period).copy_(t.view(1, period).expand(1 << 16, period))
        full[1 << 32:] = t[:77]
        return full

    want_c = one.clone().requires_grad_()
    want = nd_linear_sample(data, want_c)
    want_g, = torch.autograd.grad(want, want_c, gone)
    coord = spread(one).requires_grad_()
    out = nd_linear_sample(data, coord)
    for full, part in ((out, want), (torch.autograd.grad(out, coord, spread(gone))[0], want_g)):
        full, part = full.detach(), part.detach()
        assert torch.equal(full[1 << 32:], part[:77])
        for rows in full[:1 << 32].view(-1, period).split(1 << 13):
            assert bool((rows == part.view(1, period)).all())


@pytest.mark.parametrize("C", [1, 3, 15, 16])
@pytest.mark.parametrize("shape,most", [((64,), 5555), ((7, 7), 4878), ((4, 4, 4), 4347), ((30,), 9090), ((2, 3, 2), 8000)])
def test_tiny_volumes_around_the_most_points_of_the_one_launch_gradients(shape, most, C):
    for B in (most, most + 1):
        data, coord, gout = _inputs(shape, C, B, seed=55, dtype=torch.float32)
        for a, w in zip(_run(data, coord, gout), _oracle(data, coord, gout, np.float64)):
            assert rel_err(a, w) < 1e-5
