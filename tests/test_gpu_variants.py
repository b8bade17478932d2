"""Kernel variants that the dispatch picks by itself and that the sizes of the other tests do not reach: pairs of different tiles
in the combined backward launches, the stochastic forms of every channel tile, the wide linear kernels' ends of range, the
general convolution kernel behind a prepared data-gradient filter and behind the re-laid weight gradient."""
import ctypes

import pytest
import torch

import test_gpu_kernels as base

pytestmark = pytest.mark.gpu
ri8 = base.ri8


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


# data gradient on 32 x 32 tiles with an update on 64 x 64 and 128 x 128 ones, on 64 x 64 with 32 x 32 and 128 x 128; rows that
# start on 16-byte boundaries and others
@pytest.mark.parametrize("case", [(20, 320, 1024), (20, 300, 1000), (20, 1024, 2560), (20, 1030, 2300), (1024, 16, 512), (1030, 20, 510),
                                  (512, 1024, 2560)])
def test_linear_backward_of_two_tiles(dev, case, monkeypatch):
    base.test_linear_backward_together(dev, case, "", monkeypatch)


# N, H, W, C, K, filter, padding: the data gradient on 32 x 32 tiles with slices of the weight gradient on 64 x 64, 128 x 128; on
# 64 x 64 with 32 x 32; on 128 x 64 with 32 x 32, with 64 x 64, and with whole 64 x 64
@pytest.mark.parametrize("case", [(123, 5, 5, 16, 16, 3, 1), (9, 26, 26, 16, 80, 5, 2), (13, 27, 27, 16, 16, 3, 1), (41, 26, 26, 16, 16, 1, 0),
                                  (56, 19, 19, 16, 16, 1, 0), (60, 33, 33, 16, 48, 1, 0)])
def test_conv_backward_of_two_tiles(dev, case, monkeypatch):
    base.test_conv_backward_together(dev, case, "", monkeypatch)


# N, side, C, K with the channel tile pinned: every map's 128-channel tile, 64 channels of 4 x 4 maps, workgroups of 512 pixels
# of 16 x 16 maps (forward and data gradient)
@pytest.mark.parametrize("tile,case", [("128", (2, 32, 16, 160)), ("128", (2, 16, 32, 144)), ("128", (4, 8, 32, 144)), ("128", (16, 4, 16, 144)),
                                       ("64", (16, 4, 32, 128)), ("64", (260, 16, 16, 128)), ("64", (260, 16, 128, 16))])
def test_conv_sto_tiles(dev, tile, case, monkeypatch):
    monkeypatch.setenv("NITI_HALO_KT", tile)
    base.test_conv_requant_sto(dev, case, "floor")


# N, side, C, K: the kernel of 64-channel slices in each of its forms (channel tile, workgroups per compute unit it is made for) on
# every map (tiles of 32 channels: of at most 16 x 16): one to five slices, a last one of 48 channels, a last tile of 16 outputs,
# batches that end inside a tile (five more images); int32, rounded, the mask, both filter copies and the pooling's backward pass where the
# outputs are an even number of 32-channel slices too, StoShift
@pytest.mark.parametrize("tile,per_cu", [("32", "1"), ("64", "1"), ("64", "2"), ("128", "1"), ("128", "2")])
@pytest.mark.parametrize("case", [(2, 32, 64, 144), (1, 32, 304, 64), (3, 16, 112, 80), (3, 16, 112, 64), (2, 16, 64, 192), (4, 8, 256, 192), (16, 4, 64, 272),
                                  (32, 4, 192, 128)])
def test_conv_slices_of_64(dev, case, tile, per_cu, monkeypatch):
    monkeypatch.setenv("NITI_HALO_K64", "1")
    monkeypatch.setenv("NITI_HALO_KT", tile)
    monkeypatch.setenv("NITI_HALO_PER_CU", per_cu)
    N, Q, C, K = case
    base.test_conv_halo_tiles(dev, case, tile)
    if Q < 32:
        base.test_conv_dgrad_requant_unpool(dev, (N, Q, K, C))
    base.test_conv_requant_sto(dev, case, "floor")
    from niti_amd import ops
    from oracle import niti_oracle as po
    g = torch.Generator().manual_seed(N)
    x, w = ri8(g, N + 5, Q, Q, C), ri8(g, K, 3, 3, C)
    ref, sh_ref = po.act_calc(po.conv2d_fprop_i32(x, w, 1, 1), 0)
    y8, sh, sync = ops.conv2d_fprop_requant(x.to(dev), w.to(dev), relu=True, any_shape=True)
    assert int(sync.cpu()[1]) == 0 and torch.equal(y8.cpu(), ref.clamp(min=0)) and int(sh.cpu()) == sh_ref


# N, side, C, K: more tiles of the same kernel than the device holds workgroups at once, which take several of them in turn
# (tiles of 128 channels, of 64 on small maps; the layers' data gradients where the forward pass has an odd number of 32-channel
# slices): right, wrong and absurd predictions, StoShift, and nearly every tile stored again
MORE_THAN_FIT = [(65, 32, 64, 144), (172, 16, 272, 64), (2052, 8, 64, 64)]


@pytest.mark.parametrize("case", MORE_THAN_FIT)
def test_conv_slices_of_64_on_a_grid_larger_than_the_device(dev, case, monkeypatch):
    monkeypatch.setenv("NITI_HALO_K64", "1")
    base.test_conv_requant_predicted_shift(dev, case)


@pytest.mark.parametrize("case", MORE_THAN_FIT)
def test_conv_slices_of_64_on_a_grid_larger_than_the_device_sto(dev, case, monkeypatch):
    monkeypatch.setenv("NITI_HALO_K64", "1")
    base.test_conv_requant_sto(dev, case, "floor")


# N, side of the pooled map, channels, reduction
@pytest.mark.parametrize("case", [(172, 16, 272, 64), (2052, 8, 64, 64)])
def test_conv_slices_of_64_unpooling_on_a_grid_larger_than_the_device(dev, case, monkeypatch):
    monkeypatch.setenv("NITI_HALO_K64", "1")
    base.test_conv_dgrad_requant_unpool(dev, case)


@pytest.mark.parametrize("forward", [True, False])
def test_conv_slices_of_64_stored_again(dev, forward, monkeypatch):
    """One image with large values among images of tiny ones: nearly every tile that is stored before the range is known is computed again, with the pooled
    output, with the mask of a ReLU below and from both filter copies."""
    from niti_amd import ops
    from oracle import c_oracle as co
    from oracle import niti_oracle as po
    monkeypatch.setenv("NITI_HALO_K64", "1")
    N, Q, C, K = 65, 32, 64, 144
    base._say("conv_slices_of_64_stored_again", forward)
    g = torch.Generator().manual_seed(6161)
    x = ri8(g, N, Q, Q, C, lo=-1, hi=1)
    x[31] = ri8(g, Q, Q, C)
    if forward:
        w = ri8(g, K, 3, 3, C)
        acc = po.conv2d_fprop_i32(x, w, 1, 1)
        ref, sh_ref = po.act_calc(acc, 0)
        pooled = torch.empty((N, Q // 2, Q // 2, K), dtype=torch.int8, device=dev)
        y, sh, sync = ops.conv2d_fprop_requant(x.to(dev), w.to(dev), relu=True, pool_out=pooled)
        assert int(sync.cpu()[1]) == 0 and int(sync.cpu()[0]) == po.absmax(acc) and int(sh.cpu()) == sh_ref
        assert torch.equal(y.cpu(), ref.clamp(min=0)) and torch.equal(pooled.cpu(), po.maxpool_fwd(ref.clamp(min=0)))
        return
    w = ri8(g, C, 3, 3, K)          # the error map has C channels, the result K
    acc = co.conv_dgrad(x, w, Q, Q, 1, 1)
    ref, sh_ref = po.err_calc(acc)
    mask = ri8(g, N, Q, Q, K)
    wf = ops.conv_filter_prepare(w.to(dev), N, Q, Q)
    for kw in (dict(), dict(forward_filter=wf)):
        y, sh, sync = ops.conv2d_dgrad_requant(x.to(dev), w.to(dev), relu_mask=mask.to(dev), **kw)
        assert int(sync.cpu()[1]) == 0 and int(sh.cpu()) == sh_ref
        assert torch.equal(y.cpu(), torch.where(mask > 0, ref, torch.zeros_like(ref)))


# N, side, C, K: two to five tiles for a workgroup, some with one fewer, the last tile of channels ragged, with 64 and 128 channels
# and 256 and 512 pixels, by the kernels of 64-channel and of 32-channel slices
@pytest.mark.parametrize("case", [(2052, 8, 64, 192), (151, 32, 64, 400), (601, 32, 96, 64), (259, 16, 32, 512), (4112, 4, 128, 272)])
def test_conv_tiles_in_turns(dev, case):
    """Predictions that fit, that fit no tile and that fit some, and none: forward with the pooled output, data gradient from both filter
    copies with a mask, against the int32 results rounded by the oracle."""
    from niti_amd import ops
    from oracle import niti_oracle as po
    N, Q, C, K = case
    base._say("conv_tiles_in_turns", case)
    g = torch.Generator().manual_seed(N + K)
    x, w = ri8(g, N, Q, Q, C).to(dev), ri8(g, K, 3, 3, C).to(dev)
    x[N // 2:] //= 4          # the later images need two bits fewer
    e, mask = ri8(g, N, Q, Q, C).to(dev), ri8(g, N, Q, Q, K).to(dev)
    wb = ri8(g, C, 3, 3, K).to(dev)
    acc, dacc = ops.conv2d_fprop(x, w, 1, 1).cpu(), ops.conv2d_dgrad(e, wb, 1, 1).cpu()
    (ref, sh_ref), (dref, dsh) = po.act_calc(acc, 0), po.err_calc(dacc)
    dref = torch.where(mask.cpu() > 0, dref, torch.zeros_like(dref))
    wf = ops.conv_filter_prepare(wb, N, Q, Q)
    for off in (None, 0, 3, -2):
        def state(right):
            return {} if off is None else dict(shift_out=torch.tensor([max(right + off, 0)], dtype=torch.int32, device=dev), shift_hint=True)
        pooled = torch.empty((N, Q // 2, Q // 2, K), dtype=torch.int8, device=dev)
        y, sh, sync = ops.conv2d_fprop_requant(x, w, relu=True, pool_out=pooled, **state(sh_ref))
        assert int(sync.cpu()[1]) == 0 and int(sync.cpu()[0]) == po.absmax(acc) and int(sh.cpu()) == sh_ref
        assert torch.equal(y.cpu(), ref.clamp(min=0)) and torch.equal(pooled.cpu(), po.maxpool_fwd(ref.clamp(min=0)))
        for kw in (dict(), dict(forward_filter=wf)):
            d, sh, sync = ops.conv2d_dgrad_requant(e, wb, relu_mask=mask, **kw, **state(dsh))
            assert int(sync.cpu()[1]) == 0 and int(sh.cpu()) == dsh and torch.equal(d.cpu(), dref)
    y, sh, sync = ops.conv2d_fprop_requant(x[:-1].contiguous(), w, relu=True, any_shape=True)   # the last tile of pixels not full
    ref, sh_ref = po.act_calc(acc[:-1], 0)
    assert int(sync.cpu()[1]) == 0 and int(sh.cpu()) == sh_ref and torch.equal(y.cpu(), ref.clamp(min=0))


# more 128-channel workgroups than compute units, fewer 64-channel ones than twice those: an odd number of 64-channel groups, the last
# of 32 and of 64 channels; forward, then data gradient
@pytest.mark.parametrize("case", [(130, 16, 64, 160), (130, 16, 160, 64), (344, 8, 64, 320)])
def test_conv_slices_of_64_two_workgroups_per_unit(dev, case, monkeypatch):
    monkeypatch.setenv("NITI_HALO_K64", "1")
    base.test_conv_halo_tiles(dev, case, "auto")


# a single slice of 64 channels, the last sixteen of one channel count empty: at most one workgroup per unit, more of them, one of 128
# channels where two of 64 would be on a unit (also as the reduction of a data gradient), a grid that fits on the device with 128 channels
# only
@pytest.mark.parametrize("case", [(3, 16, 48, 64), (129, 16, 48, 96), (130, 16, 64, 128), (130, 16, 128, 64), (520, 8, 64, 256)])
def test_conv_single_slice_of_64(dev, case):
    base.test_conv_halo_tiles(dev, case, "auto")


# two slices whose int32 results come from two narrow workgroups per unit, forward and data gradient
@pytest.mark.parametrize("case", [(130, 16, 128, 128), (130, 16, 192, 96), (130, 16, 96, 192)])
def test_conv_slices_of_64_int32_from_narrow_workgroups(dev, case):
    base.test_conv_halo_tiles(dev, case, "auto")


# one to three 512-step chunks, 32 x 32 and 64 x 64 tiles, more tiles than compute units
@pytest.mark.parametrize("case", [(1, 8, 64, 64), (2, 16, 112, 48), (40, 4, 160, 32), (9, 32, 32, 64), (40, 2, 64, 96)])
def test_few_images_sto(dev, case, monkeypatch):
    """StoShift on supplied integers in a forward pass of few images, with the pooling behind the layer, by both kernels that the
    estimate chooses between."""
    from niti_amd import _lib
    from oracle import c_oracle as co
    from oracle import niti_oracle as po
    N, Q, C, K = case
    g = torch.Generator().manual_seed(12200 + N + Q + C)
    x, w = ri8(g, N, Q, Q, C), ri8(g, K, 3, 3, C)
    acc = co.conv_fprop(x, w, 1, 1)
    u = torch.randint(0, 2 ** max(po.RangeEstimate(acc) - 7, 1), acc.shape, generator=g, dtype=torch.int32)
    ref = torch.clamp(po.act_calc(acc, 0, "sto", "floor", u)[0], min=0)
    scalar = lambda v: torch.tensor([v], dtype=torch.int32, device=dev)
    for pin in ("0", "1"):
        monkeypatch.setenv("NITI_FPROP_SMALL", pin)
        for pool in (False, True):
            y, _, pooled = _lib.host().conv_layer_forward(True, x.to(dev), w.to(dev), 1, 1, True, 7, _lib.ROUND["sto"], _lib.DIV["floor"], _lib.BW["int"],
                                                          True, scalar(0), scalar(-3), scalar(1), None, pool, u.to(dev), True)
            assert torch.equal(y.cpu(), ref), (pin, pool)
            assert pooled is None or torch.equal(pooled.cpu(), po.maxpool_fwd(ref)), pin


# the kernel of 32-channel slices on an even number of them, which the dispatch gives to the other one
@pytest.mark.parametrize("tile", ["auto", "32", "64", "128"])
@pytest.mark.parametrize("case", [(2, 32, 64, 144), (3, 16, 128, 80), (8, 8, 256, 64), (16, 4, 64, 272)])
def test_conv_slices_of_32_in_pairs(dev, case, tile, monkeypatch):
    monkeypatch.setenv("NITI_HALO_K64", "0")
    if tile != "auto":
        monkeypatch.setenv("NITI_HALO_KT", tile)
    N, Q, C, K = case
    base.test_conv_halo_tiles(dev, case, tile)
    if Q < 32:
        base.test_conv_dgrad_requant_unpool(dev, (N, Q, K, C))
    base.test_conv_requant_sto(dev, case, "trunc")


# more 32-channel tiles than the device has units, and more than it holds at once (the pin is left aside), by both kernels
@pytest.mark.parametrize("k64", ["0", "1"])
@pytest.mark.parametrize("case", [(100, 16, 64, 128), (150, 16, 64, 128)])
def test_conv_pinned_to_the_narrowest_tile(dev, case, k64, monkeypatch):
    from niti_amd import ops
    from oracle import niti_oracle as po
    N, Q, C, K = case
    monkeypatch.setenv("NITI_HALO_KT", "32")
    monkeypatch.setenv("NITI_HALO_K64", k64)
    monkeypatch.setenv("NITI_HALO_PER_CU", "1")
    g = torch.Generator().manual_seed(N)
    x, w = ri8(g, N, Q, Q, C).to(dev), ri8(g, K, 3, 3, C).to(dev)
    ref, sh_ref = po.act_calc(ops.conv2d_fprop(x, w, 1, 1).cpu(), 0)
    y, sh, sync = ops.conv2d_fprop_requant(x, w)
    assert int(sync.cpu()[1]) == 0 and int(sh.cpu()) == sh_ref and torch.equal(y.cpu(), ref)


@pytest.mark.parametrize("case", [(3, 2, 32, 48), (1, 16, 48, 32)])
def test_conv_dgrad_i32_from_the_forward_copy(dev, case):
    from niti_amd import ops
    from oracle import c_oracle as co
    N, Q, C, K = case
    g = torch.Generator().manual_seed(31 + N)
    e, w = ri8(g, N, Q, Q, K), ri8(g, K, 3, 3, C)
    got = ops.conv2d_dgrad(e.to(dev), w.to(dev), forward_filter=ops.conv_filter_prepare(w.to(dev), N, Q, Q))
    assert torch.equal(got.cpu(), co.conv_dgrad(e, w, Q, Q, 1, 1))


@pytest.mark.parametrize("tile", ["0", "1", "2"])
@pytest.mark.parametrize("case", [(33, 48, 80), (65, 16, 208), (130, 80, 144)])
def test_linear_dgrad_of_aligned_rows(dev, case, tile, monkeypatch):
    """Widths that are multiples of 16 and not of 32: the kernel for any extents, rows on 16-byte boundaries."""
    from niti_amd import ops
    from oracle import niti_oracle as po
    monkeypatch.setenv("NITI_ANY_TILE", tile)
    M, O, F = case
    g = torch.Generator().manual_seed(M)
    err, w = ri8(g, M, O, lo=-60, hi=60), ri8(g, O, F)
    for method in ("round", "psto"):
        y, sh, sync = ops.linear_dgrad_requant(err.to(dev), w.to(dev), 7, method)
        ref, sh_ref = po.err_calc(po.int8mm(err, w), method, "floor")
        assert torch.equal(y.cpu(), ref) and int(sh.cpu()) == sh_ref and int(sync.cpu()[1]) == 0


@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)])
def test_gemm_f32_epilogue_of_a_split_reduction(dev, ta, tb):
    """The whole-line kernel with the reduction split over workgroups: the round trip happens where the parts are added."""
    base.test_gemm_f32_epilogue_above_2_24(dev, ta, tb, (128, 128, 8192))


# M, O, F: layers whose update would be more 128 x 128 tiles than are resident at once - few outputs and very many features, one
# with as many workgroups as are resident, a ragged last tile, the widest square of them
@pytest.mark.parametrize("case", [(5, 32, 131072), (7, 16, 100000), (3, 1024, 8192)])
def test_linear_update_of_wide_layers(dev, case):
    from niti_amd import ops
    from oracle import niti_oracle as po
    M, O, F = case
    base._say("linear_update_of_wide_layers", case)
    g = torch.Generator().manual_seed(O)
    err, act, w = ri8(g, M, O, lo=-60, hi=60), ri8(g, M, F), ri8(g, O, F)
    assert ops.linear_sync_words("wgrad", M, O, F) > 0
    acc = po.int8mm(err.t().contiguous(), act)
    rand = torch.randint(0, 1 << 24, acc.shape, generator=g, dtype=torch.int32)
    for method in ("psto", "sto"):
        low = rand & ((1 << max(po.bitwidth_int(po.absmax(acc)) - 5, 0)) - 1)
        wd = w.to(dev)
        g8, sh, sync = ops.linear_wgrad_update(err.to(dev), act.to(dev), wd, 5, method, rand=rand.to(dev) if method == "sto" else None, want_grad=True)
        ref, sh_ref = po.grad_calc(acc, 5, method, "floor", rand=low if method == "sto" else None)
        assert torch.equal(g8.cpu(), ref) and int(sh.cpu()) == sh_ref and int(sync.cpu()[1]) == 0, method
        assert torch.equal(wd.cpu(), po.weight_update(w, ref)), method


# M, O, F: both gradients as one launch of a workgroup per compute unit - one tile of dx for a quarter of the workgroups, ragged last
# tiles of both, as many tiles of dx as workgroups (the second with two chunks of samples); one row more: two launches
@pytest.mark.parametrize("case", [(1, 1024, 8192), (40, 1152, 6272), (128, 1024, 8192), (256, 2048, 4096), (129, 1024, 8192)])
def test_linear_backward_of_wide_layers(dev, case):
    from niti_amd import _lib, ops
    from oracle import niti_oracle as po
    M, O, F = case
    base._say("linear_backward_of_wide_layers", case)
    assert (_lib.lib().niti_linear_i8_backward_sync_words(M, O, F) > 0) == (M != 129)
    g = torch.Generator().manual_seed(O + M)
    err, act, w = ri8(g, M, O, lo=-60, hi=60), ri8(g, M, F), ri8(g, O, F)
    exps = [torch.tensor([e], dtype=torch.int32, device=dev) for e in (-3, -9, -2)]
    acc_e, acc_g = po.int8mm(err, w), po.int8mm(err.t().contiguous(), act)
    for err_method, grad_method, div in (("round", "psto", "floor"), ("sto", "sto", "trunc")):
        drawn = []
        for acc, bits, method in ((acc_e, 7, err_method), (acc_g, 5, grad_method)):   # wide integers, their low bits for the oracle
            u = torch.randint(0, 1 << 24, acc.shape, generator=g, dtype=torch.int32)
            low = u & ((1 << max(po.bitwidth_int(po.absmax(acc)) - bits, 0)) - 1)
            drawn.append((u.to(dev), low) if method == "sto" else (None, None))
        wd = w.to(dev)
        dx, ee, g8, _, sh, ge = ops.linear_backward(err.to(dev), act.to(dev), wd, 7, err_method, 5, grad_method, div, err_rand=drawn[0][0],
                                                    grad_rand=drawn[1][0], want_grad=True, exp_err=exps[0], exp_w=exps[1], exp_act=exps[2])
        e_ref, e_shift = po.err_calc(acc_e, err_method, div, rand=drawn[0][1])
        g_ref, g_shift = po.grad_calc(acc_g, 5, grad_method, div, rand=drawn[1][1])
        assert torch.equal(dx.cpu(), e_ref) and int(ee.cpu()) == e_shift - 12, err_method
        assert torch.equal(g8.cpu(), g_ref) and int(sh.cpu()) == g_shift and int(ge.cpu()) == g_shift + e_shift - 14, grad_method
        assert torch.equal(wd.cpu(), po.weight_update(w, g_ref)), grad_method


def test_linear_forward_of_two_sample_tiles(dev):
    """128 rows, a reduction that is no multiple of 128: two tiles of 16 samples per workgroup."""
    from niti_amd import ops
    from oracle import niti_oracle as po
    M, O, F = 128, 1024, 144
    g = torch.Generator().manual_seed(77)
    act, w = ri8(g, M, F), ri8(g, O, F)
    y, sh, sync = ops.linear_fwd_requant(act.to(dev), w.to(dev))
    ref, _ = po.act_calc(po.int8mm(act, w.t().contiguous()), 0)
    assert torch.equal(y.cpu(), ref) and int(sync.cpu()[1]) == 0


# M, O, F on both sides of one workgroup per compute unit, with whole lines and without
@pytest.mark.parametrize("case", [(64, 1024, 256), (65, 1024, 256), (128, 1024, 256), (129, 1024, 256), (64, 1000, 144), (80, 1000, 144)])
def test_linear_forward_of_operands_that_start_anywhere(dev, case):
    from niti_amd import ops
    from oracle import niti_oracle as po
    M, O, F = case
    g = torch.Generator().manual_seed(M + F)
    act, w = ri8(g, M, F), ri8(g, O, F)
    ref, _ = po.act_calc(po.int8mm(act, w.t().contiguous()), 0)

    def placed(t, offset):
        flat = torch.zeros(t.numel() + 16, dtype=torch.int8, device=dev)
        view = flat[offset:offset + t.numel()].view(t.shape)
        view.copy_(t)
        return view
    for a, b in ((0, 0), (1, 0), (0, 4), (8, 3)):
        y, sh, sync = ops.linear_fwd_requant(placed(act, a), placed(w, b))
        assert torch.equal(y.cpu(), ref) and int(sync.cpu()[1]) == 0, (a, b)


# N, H, W, C, K, filter, padding: whole 128-byte steps of one tap; 512- and 256-pixel tiles; a filter of more than 32 taps
@pytest.mark.parametrize("case", [(2, 9, 9, 32, 128, 3, 1), (128, 30, 30, 32, 16, 3, 1), (32, 30, 30, 144, 16, 3, 1), (1, 9, 9, 16, 16, 7, 3)])
def test_conv_dgrad_from_its_own_copy(dev, case):
    """The data gradient from a filter flipped beforehand, on maps outside the 3 x 3 kernels': the general convolution kernel."""
    from niti_amd import ops
    from oracle import c_oracle as co
    from oracle import niti_oracle as po
    N, H, W, C, K, R, pad = case
    base._say("conv_dgrad_from_its_own_copy", case)
    g = torch.Generator().manual_seed(51 + N)
    e, w = ri8(g, N, H + 2 * pad - R + 1, W + 2 * pad - R + 1, K), ri8(g, K, R, R, C)
    ref = co.conv_dgrad(e, w, H, W, 1, pad)
    copy = ops.conv_filter_prepare(w.to(dev), N, H, W, 1, pad, dgrad=True)
    am = ops.new_scalar_u32(dev)
    assert torch.equal(ops.conv2d_dgrad(e.to(dev), w.to(dev), 1, pad, absmax=am, prepared_filter=copy).cpu(), ref)
    assert int(am.cpu()) == po.absmax(ref)


# N, H, W, C, K: filters that are no multiple of 16, so both operands are re-laid; batches of whole 128-byte steps with few and many
# channels, shorter ones with 256- and 512-row tiles
@pytest.mark.parametrize("case", [(128, 4, 4, 16, 10), (128, 4, 4, 1600, 10), (64, 4, 4, 3200, 10), (16, 4, 4, 6400, 10)])
def test_conv_wgrad_re_laid(dev, case):
    from niti_amd import ops
    from oracle import c_oracle as co
    from oracle import niti_oracle as po
    N, H, W, C, K = case
    base._say("conv_wgrad_re_laid", case)
    g = torch.Generator().manual_seed(61 + C)
    a, e = ri8(g, N, H, W, C), ri8(g, N, H, W, K, lo=-40, hi=40)
    ref = co.conv_wgrad(a, e, 3, 3, 1, 1)
    am = ops.new_scalar_u32(dev)
    assert torch.equal(ops.conv2d_wgrad(a.to(dev), e.to(dev), 3, 3, absmax=am).cpu(), ref) and int(am.cpu()) == po.absmax(ref)


def test_quantiser_entries_of_the_c_abi(dev):
    """The two entries that the front end does not call, against the one it does."""
    from niti_amd import _lib as L
    from niti_amd import ops
    x = torch.randn((9, 3, 16, 16), generator=torch.Generator().manual_seed(4)).to(dev)
    want, exp = ops.quantize_input(x)
    N, C, H, W = x.shape
    stream = torch.cuda.current_stream().cuda_stream
    y, e = torch.full_like(want, 55), torch.full_like(exp, 55)
    word = torch.zeros(1, dtype=torch.int32, device=dev)
    L.check(L.lib().niti_quantize_f32_i8(x.data_ptr(), y.data_ptr(), N, C, H, W, 16, 7, word.data_ptr(), e.data_ptr(), stream), "quantize")
    assert torch.equal(y, want) and torch.equal(e, exp)
    y.fill_(55), e.fill_(55)
    parts = torch.empty(256, dtype=torch.int32, device=dev)
    target = torch.arange(9, device=dev)
    copied = torch.zeros_like(target)
    L.check(L.lib().niti_quantize_batch_f32_i8(x.data_ptr(), y.data_ptr(), N, C, H, W, 16, 7, parts.data_ptr(), e.data_ptr(), target.data_ptr(),
                                               copied.data_ptr(), 9, ctypes.c_void_p(stream)), "quantize_batch")
    assert torch.equal(y, want) and torch.equal(e, exp) and torch.equal(copied, target)


# batches on both sides of the line between workgroups of half an image and of a whole one, every number of filters and of channels
@pytest.mark.parametrize("case", [(1, 32, 3), (42, 32, 1), (43, 64, 3), (42, 64, 2), (42, 128, 3), (43, 128, 3), (2, 256, 3), (43, 256, 1)])
def test_first_layer_wgrad_by_images(dev, case):
    """The first layer's weight gradient and update, sums of both signs beyond the float32 mantissa among them."""
    from niti_amd import ops
    from oracle import c_oracle as co
    from oracle import niti_oracle as po
    N, K, Cw = case
    base._say("first_layer_wgrad", case)
    g = torch.Generator().manual_seed(N + K)
    act, err, w = torch.zeros(N, 32, 32, 16, dtype=torch.int8), ri8(g, N, 32, 32, K), ri8(g, K, 3, 3, Cw)
    act[..., :Cw] = ri8(g, N, 32, 32, Cw)
    act[..., 0], err[..., ::2], err[..., 1::2] = 127, 127, -127
    dw = co.conv_wgrad(act, err, 3, 3, 1, 1)
    gref, sh_ref = po.grad_calc(dw, 5, "psto")
    for want_dw in (False, True):
        wd = w.to(dev)
        wide = torch.zeros(K, 3, 3, 16, dtype=torch.int8, device=dev)
        wide[..., :Cw] = wd
        prepared = ops.conv_filter_prepare(wide, N, 32, 32, 1, 1)
        g8, d, sh, sync = ops.conv2d_wgrad_update(act.to(dev), err.to(dev), wd, want_grad=True, want_dw=want_dw, prepared_filter=prepared)
        assert int(sync.cpu()[0]) == po.absmax(dw) and int(sh.cpu()) == sh_ref
        assert torch.equal(g8.cpu(), gref[..., :Cw]) and torch.equal(wd.cpu(), po.weight_update(w, gref[..., :Cw].contiguous()))
        wide[..., :Cw] = wd
        assert torch.equal(prepared, ops.conv_filter_prepare(wide, N, 32, 32, 1, 1))
        assert not want_dw or torch.equal(d.cpu(), dw)


# N, side, C, K of layers whose two gradients run as a pair of launches.  Update beside the data gradient: its tiles of 32, 64 and 128
# channels on every map; one slice of partial sums and 67, three input-channel groups of 64, batches that end inside a tile; some
# workgroups for the update fewer than the device has units.  Update by workgroups that multiply as well: 64 and 128 channels, and
# more of them than the device has units; by some that multiply several tiles.
PAIRS = [(3, 16, 64, 128), (5, 8, 192, 128), (2, 8, 256, 512), (5, 32, 64, 128), (70, 16, 128, 128), (70, 8, 512, 128), (36, 32, 128, 192), (70, 16, 256, 128),
         (300, 8, 256, 128), (97, 32, 128, 128), (115, 32, 64, 128), (115, 32, 128, 128), (230, 16, 256, 128), (900, 8, 256, 128), (150, 16, 256, 256),
         (135, 32, 128, 128), (1030, 8, 192, 128)]


@pytest.mark.parametrize("case", PAIRS)
def test_conv_backward_pair(dev, case, monkeypatch):
    """Both gradients of a 3x3 layer as the weight gradient's sums and the data gradient along with the update: error, mask and
    pooling as in the one launch, exponents, weights, filter copy, with right, wrong and no predicted shifts."""
    from niti_amd import _lib, ops
    from oracle import c_oracle as co
    from oracle import niti_oracle as po
    N, Q, C, K = case
    monkeypatch.setenv("NITI_BACKWARD_PAIR", "1")
    base._say("conv_backward_pair", case)
    assert _lib.lib().niti_conv2d_i8_backward_pair_sync_words(N, Q, Q, C, K, 3, 3, 1) > 0
    g = torch.Generator().manual_seed(9800 + N + Q + C + K)
    x, w, e = ri8(g, N, Q, Q, C), ri8(g, K, 3, 3, C), ri8(g, N, Q, Q, K, lo=-40, hi=40)
    scalar = lambda v: torch.tensor([v], dtype=torch.int32, device=dev)
    dacc, wacc = co.conv_dgrad(e, w, Q, Q, 1, 1), co.conv_wgrad(x, e, 3, 3, 1, 1)
    whole = ri8(g, N, 2 * Q, 2 * Q, C, lo=-3, hi=4)      # few values: ties in most windows
    pooled = po.maxpool_fwd(whole)
    for kind, err_method, grad_method, off in (("plain", "round", "psto", None), ("mask", "round", "psto", 0), ("mask", "psto", "round", 1), ("first", "round", "psto", -1)):
        dref, dsh = po.err_calc(dacc, err_method)
        gref, gsh = po.grad_calc(wacc, 5, grad_method)
        if kind == "mask":
            dref = dref * (x > 0)
        elif kind == "first":
            dref = po.maxpool_bwd(pooled, dref * (pooled > 0), whole, ties=kind)
        wd = w.to(dev)
        prepared = ops.conv_filter_prepare(wd, N, Q, Q, 1, 1)
        guess = [None, None] if off is None else [scalar(dsh + off), scalar(gsh + off)]
        dx, de, unpooled, g8, _, sh, ge, one = ops.conv2d_backward(
            e.to(dev), x.to(dev), wd, err_method=err_method, grad_method=grad_method, relu_mask=None if kind == "plain" else (pooled if kind == "first" else x).to(dev),
            pool_in=whole.to(dev) if kind == "first" else None, want_grad=True, exp_err=scalar(-4), exp_w=scalar(-3), exp_act=scalar(2), prepared_filter=prepared,
            err_shift=guess[0], grad_shift=guess[1])
        assert one and unpooled == (kind == "first")
        assert torch.equal(dx.cpu(), dref) and int(de.cpu()) == dsh - 7, (kind, off)
        assert torch.equal(g8.cpu(), gref) and int(sh.cpu()) == gsh and int(ge.cpu()) == gsh + dsh - 7 + 2, (kind, off)
        assert off is None or (int(guess[0].cpu()), int(guess[1].cpu())) == (dsh, gsh)
        assert torch.equal(wd.cpu(), po.weight_update(w, gref)), (kind, off)
        assert torch.equal(prepared, ops.conv_filter_prepare(wd, N, Q, Q, 1, 1)), (kind, off)
    assert not ops.sync_arena.timed_out(dev)


# few pixels or short sums of many channels, on either side of the lines
@pytest.mark.parametrize("case,pair", [((37, 8, 1792, 128), False), ((43, 8, 768, 320), False), ((9, 16, 1728, 128), False), ((44, 8, 448, 576), True),
                                       ((128, 8, 576, 128), True), ((128, 32, 128, 128), True)])
def test_conv_backward_pair_rule(dev, case, pair, monkeypatch):
    from niti_amd import _lib
    N, Q, C, K = case
    for name in ("NITI_BACKWARD_PAIR", "NITI_BACKWARD_TOGETHER"):
        monkeypatch.delenv(name, raising=False)
    assert (_lib.lib().niti_conv2d_i8_backward_pair_sync_words(N, Q, Q, C, K, 3, 3, 1) > 0) == pair


@pytest.mark.parametrize("case", [(12, 16, 128, 128), (115, 32, 64, 128)])
def test_conv_backward_pair_sums_beyond_2_23(dev, case, monkeypatch):
    """Partial sums that need more than 24 bits, from some workgroups of the weight gradient and not from others."""
    from niti_amd import ops
    from oracle import c_oracle as co
    from oracle import niti_oracle as po
    N, Q, C, K = case
    monkeypatch.setenv("NITI_BACKWARD_PAIR", "1")
    monkeypatch.setenv("NITI_WGRAD_BLOCKS", "16")
    base._say("conv_backward_pair, partial sums > 2^23", case)
    g = torch.Generator().manual_seed(4500 + Q)
    act, err, w = ri8(g, N, Q, Q, C, lo=-20, hi=20), ri8(g, N, Q, Q, K, lo=-20, hi=20), ri8(g, K, 3, 3, C)
    n_hot = N // 4
    act[:n_hot, :, :, :32] = 127
    err[:n_hot] = 127
    err[:n_hot, :, :, 1::2] = -127
    dw = co.conv_wgrad(act, err, 3, 3, 1, 1)
    assert int(dw.abs().max()) > 2 ** 23 and int(dw[:, :, :, 32:].abs().max()) < 2 ** 22
    gref, gsh = po.grad_calc(dw, 5, "psto")
    wd = w.to(dev)
    prepared = ops.conv_filter_prepare(wd, N, Q, Q, 1, 1)
    g8, sh = ops.conv2d_backward(err.to(dev), act.to(dev), wd, want_grad=True, prepared_filter=prepared)[3:6:2]
    assert torch.equal(g8.cpu(), gref) and int(sh.cpu()) == gsh and torch.equal(wd.cpu(), po.weight_update(w, gref))
    assert torch.equal(prepared, ops.conv_filter_prepare(wd, N, Q, Q, 1, 1))


# the update beside the data gradient, by workgroups that multiply one tile as well, by those that multiply several; filters that leave
# part of the last 64 and of the last 128 empty
@pytest.mark.parametrize("options", [dict(), dict(pool="all", div="trunc", bw="f32", want_grad=False), dict(pool="first", f32=False)])
@pytest.mark.parametrize("case", [(12, 16, 128, 112), (40, 8, 192, 240), (115, 32, 64, 112), (115, 32, 128, 240), (135, 32, 128, 176)])
def test_conv_backward_pair_options(dev, case, options, monkeypatch):
    """Partial sums beyond 24 bits from some workgroups, whole sums beyond the float32 mantissa, through the float32 epilogue and not;
    both divisions and bit widths, both tie rules of the pooling's backward pass, with and without the int8 gradient."""
    from niti_amd import ops
    from oracle import c_oracle as co
    from oracle import niti_oracle as po
    N, Q, C, K = case
    f32, div, bw, pool, want_grad = (options.get(k, v) for k, v in (("f32", True), ("div", "floor"), ("bw", "int"), ("pool", None), ("want_grad", True)))
    monkeypatch.setenv("NITI_BACKWARD_PAIR", "1")
    monkeypatch.setenv("NITI_WGRAD_BLOCKS", "16")
    base._say("conv_backward_pair options", case, options)
    g = torch.Generator().manual_seed(5600 + N + K)
    act, err, w = ri8(g, N, Q, Q, C, lo=-20, hi=20), ri8(g, N, Q, Q, K, lo=-20, hi=20), ri8(g, K, 3, 3, C)
    act[:N // 2, :, :, :32], err[:N // 2], err[:N // 2, :, :, 1::2] = 127, 127, -127
    dacc, wacc = co.conv_dgrad(err, w, Q, Q, 1, 1), co.conv_wgrad(act, err, 3, 3, 1, 1)
    assert int(wacc.abs().max()) > 2 ** 24 and int(wacc[:, :, :, 32:].abs().max()) < 2 ** 23 and not torch.equal(wacc, po.f32_roundtrip(wacc))
    if f32:
        dacc, wacc = po.f32_roundtrip(dacc), po.f32_roundtrip(wacc)
    (dref, dsh), (gref, gsh) = po.err_calc(dacc, div_mode=div, bw_mode=bw), po.grad_calc(wacc, 5, "psto", div_mode=div, bw_mode=bw)
    kw = {}
    if pool is not None:
        whole = ri8(g, N, 2 * Q, 2 * Q, C, lo=-3, hi=4)
        pooled = po.maxpool_fwd(whole)
        dref = po.maxpool_bwd(pooled, dref * (pooled > 0), whole, ties=pool)
        kw = dict(relu_mask=pooled.to(dev), pool_in=whole.to(dev), ties=pool)
    wd = w.to(dev)
    prepared = ops.conv_filter_prepare(wd, N, Q, Q, 1, 1)
    scalar = lambda v: torch.tensor([v], dtype=torch.int32, device=dev)
    dx, de, unpooled, g8, _, sh, ge, one = ops.conv2d_backward(
        err.to(dev), act.to(dev), wd, f32_epilogue=f32, div_mode=div, bw_mode=bw, want_grad=want_grad, prepared_filter=prepared,
        exp_err=scalar(-4), exp_w=scalar(-3), exp_act=scalar(2), **kw)
    assert one and unpooled == (pool is not None) and (g8 is not None) == want_grad
    assert torch.equal(dx.cpu(), dref) and int(de.cpu()) == dsh - 7
    assert int(sh.cpu()) == gsh and int(ge.cpu()) == gsh + dsh - 7 + 2 and (g8 is None or torch.equal(g8.cpu(), gref))
    assert torch.equal(wd.cpu(), po.weight_update(w, gref)) and torch.equal(prepared, ops.conv_filter_prepare(wd, N, Q, Q, 1, 1))
    assert not ops.sync_arena.timed_out(dev) and not ops.sync_timeouts(dev)


@pytest.mark.parametrize("case", [(3, 16, 64, 128), (115, 32, 64, 128), (135, 32, 128, 128)])
def test_conv_backward_pair_with_one_prediction(dev, case, monkeypatch):
    """A predicted shift for one of the two gradients only, right and absurd: the other one is as without any."""
    from niti_amd import ops
    from oracle import c_oracle as co
    from oracle import niti_oracle as po
    N, Q, C, K = case
    monkeypatch.setenv("NITI_BACKWARD_PAIR", "1")
    base._say("conv_backward_pair, one prediction", case)
    g = torch.Generator().manual_seed(7700 + N)
    x, w, e = ri8(g, N, Q, Q, C), ri8(g, K, 3, 3, C), ri8(g, N, Q, Q, K, lo=-40, hi=40)
    dref, dsh = po.err_calc(co.conv_dgrad(e, w, Q, Q, 1, 1))
    gref, gsh = po.grad_calc(co.conv_wgrad(x, e, 3, 3, 1, 1), 5, "psto")
    for which, right in (("err_shift", dsh), ("grad_shift", gsh)):
        for guess in (right, right + 9, -3):
            word = torch.tensor([guess], dtype=torch.int32, device=dev)
            wd = w.to(dev)
            prepared = ops.conv_filter_prepare(wd, N, Q, Q, 1, 1)
            dx, _, _, g8, _, sh, _, one = ops.conv2d_backward(e.to(dev), x.to(dev), wd, want_grad=True, prepared_filter=prepared, **{which: word})
            assert one and torch.equal(dx.cpu(), dref) and torch.equal(g8.cpu(), gref) and int(sh.cpu()) == gsh, (which, guess)
            assert int(word.cpu()) == right and torch.equal(wd.cpu(), po.weight_update(w, gref)), (which, guess)
    assert not ops.sync_arena.timed_out(dev) and not ops.sync_timeouts(dev)


def test_updates_waits_are_flagged_in_the_words_of_the_call():
    """Waits with a limit of zero in every call that updates weights beside a data gradient: the update's waits have a bit of their own
    in the flag word that sync_arena.timed_out looks at, that of the slice the call was given."""
    import os
    import subprocess
    import sys
    code = """
import os
import torch
from niti_amd import _lib, ops
dev = torch.device("cuda:0")
ri = lambda *s: torch.randint(-127, 128, s, dtype=torch.int8, device=dev)

def flags(name, call, **env):
    os.environ.update(env)
    ops.sync_arena.reset(dev)
    call()
    torch.cuda.synchronize()
    seen = 0
    for t in _lib.host().arena_flags(0):
        seen |= int(t.item())
    print("FLAGS", name, seen, int(ops.sync_arena.timed_out(dev)), flush=True)
    for k in env:
        del os.environ[k]

def conv(N, Q, C, K):
    w = ri(K, 3, 3, C)
    assert ops.conv2d_backward(ri(N, Q, Q, K), ri(N, Q, Q, C), w, prepared_filter=ops.conv_filter_prepare(w, N, Q, Q, 1, 1))[-1]

def linear(M, O, F):
    assert _lib.lib().niti_linear_i8_backward_sync_words(M, O, F) > 0
    ops.linear_backward(ri(M, O), ri(M, F), ri(O, F))

for case in ((3, 16, 64, 128), (115, 32, 128, 128), (135, 32, 128, 128)):
    flags("pair%d" % case[0], lambda: conv(*case), NITI_BACKWARD_PAIR="1")
for slices in "14":
    flags("together" + slices, lambda: conv(3, 16, 64, 128), NITI_BACKWARD_PAIR="0", NITI_BACKWARD_TOGETHER="1", NITI_ANY_SLICES=slices)
flags("linear_wide", lambda: linear(128, 1024, 8192))
flags("linear_any", lambda: linear(100, 300, 1000))
"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = subprocess.run([sys.executable, "-c", code], cwd=root, env=dict(os.environ, NITI_SYNC_TIMEOUT_MS="0"), capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stderr[-2000:]
    lines = [line.split()[1:] for line in out.stdout.splitlines() if line.startswith("FLAGS")]
    assert len(lines) == 7
    for name, seen, timed_out in lines:
        assert int(seen) & 4 and timed_out == "1", out.stdout


@pytest.mark.parametrize("case", [(3, 16, 64, 128), (115, 32, 128, 128), (135, 32, 128, 128)])
def test_conv_backward_pair_gives_up(case):
    """Waits with a limit of zero: the launch ends and the device-wide word says so."""
    import os
    import subprocess
    import sys
    code = """
import torch
from niti_amd import ops
N, Q, C, K = %r
dev = torch.device("cuda:0")
ri = lambda *s: torch.randint(-127, 128, s, dtype=torch.int8, device=dev)
w = ri(K, 3, 3, C)
ops.conv2d_backward(ri(N, Q, Q, K), ri(N, Q, Q, C), w, prepared_filter=ops.conv_filter_prepare(w, N, Q, Q, 1, 1))
torch.cuda.synchronize()
print("STICKY", int(ops.sync_timeouts(dev)))
""" % (case,)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, NITI_SYNC_TIMEOUT_MS="0", NITI_BACKWARD_PAIR="1")
    out = subprocess.run([sys.executable, "-c", code], cwd=root, env=env, capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stderr[-2000:]
    assert "STICKY 1" in out.stdout
