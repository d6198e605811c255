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
# columns and channels; K below, at and beyond the four steps loaded ahead
@pytest.mark.parametrize("h,w,cin,cout,ks,transposed", [
    (9, 7, 8, 33, 1, False), (33, 31, 64, 32, 1, False), (33, 31, 72, 40, 1, False),
    (256, 255, 24, 33, 1, False), (256, 129, 24, 40, 1, False),
    (365, 360, 8, 20, 3, False), (363, 360, 8, 32, 3, False),
    (4, 1, 16, 1, 3, False), (8, 33, 32, 33, 3, False), (64, 95, 48, 65, 3, False),
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
# others, channels below and beyond a 64-column tile, a ragged last split, the
# output gradient at fine pixels
@pytest.mark.parametrize("batch,h,w,cin,cout,ks,fine", [
    (2, 3, 4, 8, 8, 3, False), (1, 5, 12, 16, 72, 3, False), (3, 17, 20, 72, 8, 1, False),
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
