"""The bfloat16 convolution kernels on both sides of the lines at which their
tiles and paths change.  Operands are small whole numbers: every product and
every sum is exact in fp32, so the results equal torch's fp64 ones."""
import pytest

pytestmark = pytest.mark.gpu


def _ints(g, *shape):
    import torch
    return torch.randint(-2, 3, shape, generator=g).double()


# 32 x 32 tiles below 1024 wide tiles, 64 x 64 (cout > 32) and 128 x 32 from
# there on; 3 x 3 from LDS where cin % 16 == 0 and h % 4 == 0, with ragged
# columns and channels, one and two rows a wavefront; K below, at and beyond the four steps loaded ahead
@pytest.mark.parametrize("h,w,cin,cout,ks,transposed", [
    (9, 7, 8, 33, 1, False), (33, 31, 64, 32, 1, False), (33, 31, 72, 40, 1, False),
    (256, 255, 24, 33, 1, False), (256, 129, 24, 40, 1, False),
    (365, 360, 8, 20, 3, False), (363, 360, 8, 32, 3, False),
    (4, 1, 16, 1, 3, False), (8, 33, 32, 33, 3, False), (64, 95, 48, 65, 3, False),
    (256, 999, 16, 40, 3, False), (260, 999, 16, 40, 3, False),
    (128, 130, 16, 17, 1, True), (9, 5, 40, 9, 1, True)])
def test_convolution_tiles(h, w, cin, cout, ks, transposed):
    import torch
    from psvwave_amd import _lib
    lib = _lib.load()
    print(f"[conv] {h}x{w} {cin}->{cout} ks {ks} {transposed}", flush=True)
    g = torch.Generator().manual_seed(h * w + cout)
    x, b = _ints(g, 1, cin, h, w), _ints(g, cout)
    if transposed:
        wt = _ints(g, cin, cout, 2, 2)
        ref = torch.nn.functional.conv_transpose2d(x, wt, b, stride=2)
        wd = wt.permute(2, 3, 1, 0).reshape(4 * cout, cin)
    else:
        wt = _ints(g, cout, cin, ks, ks)
        ref = torch.nn.functional.conv2d(x, wt, b, padding=ks // 2)
        wd = wt.permute(0, 2, 3, 1).reshape(cout, -1)
    xd = x[0].permute(1, 2, 0).contiguous().to("cuda", torch.bfloat16)
    wd = wd.contiguous().to("cuda", torch.bfloat16)
    bd = b.float().cuda()
    out = torch.full(tuple(ref[0].permute(1, 2, 0).shape), float("nan"), device="cuda")
    _lib.check(lib.psv_conv2d_bf16(xd.data_ptr(), wd.data_ptr(), bd.data_ptr(), out.data_ptr(), 1,
                                   h, w, cin, cout, ks, int(transposed), 0, cout, 0,
                                   torch.cuda.current_stream().cuda_stream))
    assert torch.equal(out.cpu().double(), ref[0].permute(1, 2, 0))


# rows of a multiple of four pixels (one of them: both edges in a group) and
# others, channels below and beyond the tiles, ragged last splits, the
# output gradient at fine pixels
@pytest.mark.parametrize("batch,h,w,cin,cout,ks,fine", [
    (2, 3, 4, 8, 8, 3, False), (1, 5, 12, 16, 72, 3, False), (3, 17, 20, 72, 8, 1, False),
    (3, 41, 52, 64, 64, 3, False), (1, 70, 61, 64, 64, 3, False), (3, 41, 52, 16, 32, 3, False),
    (2, 40, 36, 8, 16, 3, False), (1, 31, 37, 8, 16, 3, False), (1, 7, 2, 8, 8, 3, False),
    (2, 6, 8, 16, 24, 1, True), (1, 9, 5, 16, 24, 1, True)])
def test_weight_gradient_tiles(batch, h, w, cin, cout, ks, fine):
    import torch
    from psvwave_amd import _lib
    lib = _lib.load()
    print(f"[wgrad] {batch}x{h}x{w} {cin}->{cout} ks {ks} {fine}", flush=True)
    g = torch.Generator().manual_seed(h * w + cout)
    x = _ints(g, batch, cin, h, w)
    if fine:
        wt = torch.zeros(cin, cout, 2, 2, dtype=torch.float64, requires_grad=True)
        dy = _ints(g, batch, cout, 2 * h, 2 * w)
        (torch.nn.functional.conv_transpose2d(x, wt, stride=2) * dy).sum().backward()
        ref = wt.grad.permute(2, 3, 1, 0).reshape(4 * cout, cin)
    else:
        wt = torch.zeros(cout, cin, ks, ks, dtype=torch.float64, requires_grad=True)
        dy = _ints(g, batch, cout, h, w)
        (torch.nn.functional.conv2d(x, wt, padding=ks // 2) * dy).sum().backward()
        ref = wt.grad.permute(0, 2, 3, 1).reshape(cout, -1)
    nhwc = [t.permute(0, 2, 3, 1).contiguous().to("cuda", torch.bfloat16) for t in (x, dy)]
    ws = torch.empty(1 << 20, device="cuda")
    dw = torch.full(tuple(ref.shape), float("nan"), device="cuda")
    db = torch.full((ref.shape[0],), float("nan"), device="cuda")
    _lib.check(lib.psv_conv_wgrad_bf16(nhwc[1].data_ptr(), cout, int(fine), cout,
                                       nhwc[0].data_ptr(), cin, cin, ks, batch, h, w,
                                       dw.data_ptr(), db.data_ptr(), ws.data_ptr(), ws.numel(),
                                       torch.cuda.current_stream().cuda_stream))
    assert torch.equal(dw.cpu().double(), ref)
    sums = db.cpu().double()
    sums = sums.view(4, cout).sum(0) if fine else sums
    assert torch.equal(sums, dy.sum(dim=(0, 2, 3)))


# 8 channels to a store where everything is aligned for it, one value else: the
# same bits, in each mode, with ragged rows, columns and channels, and with the
# pre-activation, the activation and the stored derivative
@pytest.mark.parametrize("h,w,cin,cout,ks,mode", [
    (8, 33, 32, 40, 3, 0), (4, 1, 16, 8, 3, 0), (5, 37, 16, 24, 3, 0), (365, 360, 8, 24, 3, 0),
    (9, 7, 8, 72, 1, 0), (257, 255, 24, 40, 1, 0), (9, 5, 40, 8, 1, 1), (130, 128, 16, 24, 1, 1),
    (6, 5, 16, 40, 1, 2)])
@pytest.mark.parametrize("f32,fused", [(0, False), (1, False), (0, True)])
def test_convolution_stores(h, w, cin, cout, ks, mode, f32, fused):
    import torch
    from psvwave_amd import _lib
    lib = _lib.load()
    print(f"[stores] {h}x{w} {cin}->{cout} ks {ks} mode {mode} f32 {f32} {fused}", flush=True)
    g = torch.Generator().manual_seed(h * w + cout)
    taps, up = (ks * ks, 1) if mode < 2 else (4, 2)
    x = torch.randn(1, up * h, up * w, cin, generator=g).to("cuda", torch.bfloat16)
    rows = 4 * cout if mode == 1 else cout
    wt = torch.randn(rows, taps * cin, generator=g).to("cuda", torch.bfloat16)
    b = torch.randn(cout, generator=g).cuda()
    oh, ow = (2 * h, 2 * w) if mode == 1 else (h, w)
    z = torch.randn(oh, ow, cout, generator=g).to("cuda", torch.bfloat16)
    results = []
    for off in (8, 4):  # in 16-byte accesses; value by value
        stride = cout + 16
        out = torch.full((oh, ow, stride), 7.0, device="cuda",
                         dtype=torch.float32 if f32 else torch.bfloat16)
        pre = torch.zeros(oh, ow, cout, device="cuda", dtype=torch.bfloat16)
        _lib.check(lib.psv_conv_bf16(
            x.data_ptr(), cin, wt.data_ptr(), b.data_ptr(), out.data_ptr(), f32, stride, off,
            pre.data_ptr() if fused and mode == 0 else 0, z.data_ptr() if fused else 0, cout, 1, h,
            w, cin, cout, ks, mode, int(fused), torch.cuda.current_stream().cuda_stream))
        assert (out[..., :off] == 7).all() and (out[..., off + cout:] == 7).all()
        results.append((out[..., off:off + cout].float().cpu(), pre.float().cpu()))
    assert torch.equal(results[0][0], results[1][0])
    assert torch.equal(results[0][1], results[1][1])


@pytest.mark.parametrize("h,w,c", [(2, 2, 8), (6, 10, 24), (34, 62, 40), (2, 130, 64)])
def test_pooling_in_wide_accesses(h, w, c):
    import torch
    from psvwave_amd import _lib
    lib = _lib.load()
    print(f"[pool] {h}x{w}x{c}", flush=True)
    g = torch.Generator().manual_seed(h * w + c)
    stream = torch.cuda.current_stream().cuda_stream
    a = _ints(g, h, w, c).to("cuda", torch.bfloat16)  # with ties
    room = torch.zeros(h * w * c + 8, device="cuda", dtype=torch.bfloat16)
    shifted = room[4:4 + h * w * c].view(h, w, c)  # 8 bytes off: value by value
    shifted.copy_(a)
    pooled = []
    for t in (a, shifted):
        out = torch.zeros(h // 2, w // 2, c, device="cuda", dtype=torch.bfloat16)
        _lib.check(lib.psv_maxpool2_bf16(t.data_ptr(), out.data_ptr(), h, w, c, stream))
        pooled.append(out.cpu())
    ref = torch.nn.functional.max_pool2d(a.float().cpu().permute(2, 0, 1)[None], 2)[0]
    assert torch.equal(pooled[0].float().permute(2, 0, 1), ref)
    assert torch.equal(pooled[0], pooled[1])
    z = torch.randn(h, w, c, generator=g).to("cuda", torch.bfloat16)
    d = torch.randn(h // 2, w // 2, c, generator=g).cuda()
    skip = torch.randn(h, w, 2 * c, generator=g).to("cuda", torch.bfloat16)
    for dpool, dskip in ((d, skip), (d, None), (None, skip)):
        grads = []
        for t in (a, shifted):
            out = torch.zeros(h, w, c, device="cuda", dtype=torch.bfloat16)
            _lib.check(lib.psv_maxpool2_backward_bf16(
                t.data_ptr(), z.data_ptr(), 0 if dpool is None else dpool.data_ptr(),
                0 if dskip is None else dskip.data_ptr(), 2 * c, c, out.data_ptr(), 1, h, w, c,
                stream))
            grads.append(out.float().cpu())
        assert torch.equal(grads[0], grads[1])


# more items than a launch holds, one value to several blocks, flipped taps,
# padded and cut channels
@pytest.mark.parametrize("half", [False, True])
def test_rearrangements(half):
    import torch
    from psvwave_amd.precond import _rearrange
    shapes = [(1, 1, 1, 1), (3, 3, 3, 8), (128, 3, 3, 40), (7, 2, 2, 512), (5, 1, 1, 9)] * 8
    results = []
    for device in ("cpu", "cuda"):
        items = []
        for n, (a, b, c, d) in enumerate(shapes):
            valid = d if n % 3 else max(1, d - 3)
            src = torch.arange(a * b * c * valid, dtype=torch.float32).mul_(0.37).add_(n)
            dst = torch.full((a, b * c * d), float("nan"), device=device,
                             dtype=torch.bfloat16 if half else torch.float32)
            flip = -1 if n % 2 else 1  # the two inner dimensions in either order
            items.append((dst, src.to(device), (b * c - 1) if flip < 0 else 0, (a, b, c, d),
                          (b * c, flip * c, flip, a * b * c), valid))
        print(f"[rearrange] {device} {half}", flush=True)
        _rearrange(items)
        results.append([item[0].float().cpu() for item in items])
    for x, y in zip(*results):
        assert torch.equal(x, y)
