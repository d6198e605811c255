"""The training layouts and gradients under a default dtype other than
float32: the kernels read and write float32 whatever torch's default is."""
import pytest

from psvwave_amd import precond

torch = pytest.importorskip("torch")


@pytest.fixture(params=["float64", "float16", "bfloat16"])
def default_dtype(request):
    before = torch.get_default_dtype()
    torch.set_default_dtype(getattr(torch, request.param))
    yield getattr(torch, request.param)
    torch.set_default_dtype(before)


def test_parameter_gradients_are_float32(default_dtype):
    trainer = precond.HipUNetTrainer.__new__(precond.HipUNetTrainer)
    trainer.device = "cpu"
    conv = torch.nn.Conv2d(8, 24, 3, dtype=torch.float32)
    ct = torch.nn.ConvTranspose2d(16, 8, 2, stride=2, dtype=torch.float32)
    dw = torch.arange(24 * 9 * 8, dtype=torch.float32).mul_(0.37).view(24, 72)
    dt = torch.arange(4 * 8 * 16, dtype=torch.float32).mul_(0.37).view(32, 16)
    grads = trainer._to_param_grads({"up": [trainer._convt_layout(ct)]},
                                    {conv: (dw, None), ct: (dt, None)})
    (_, g, _), (_, h, _) = grads
    assert g.dtype == h.dtype == torch.float32
    assert torch.equal(g, dw.view(24, 3, 3, 8).permute(0, 3, 1, 2))
    assert torch.equal(h, dt.view(2, 2, 8, 16).permute(3, 2, 0, 1))


@pytest.mark.parametrize("dst, src", [
    (torch.empty(4, 6, dtype=torch.float64), torch.zeros(24)),
    (torch.empty(4, 6, dtype=torch.float16), torch.zeros(24)),
    (torch.empty(4, 6), torch.zeros(24, dtype=torch.float64)),
    (torch.empty(4, 5), torch.zeros(24)),
    (torch.empty(6, 4).T, torch.zeros(24)),
    (torch.empty(4, 6), torch.zeros(48)[::2]),
    (torch.empty(4, 6, device="meta"), torch.zeros(24)),
])
def test_tensors_the_kernel_cannot_take_are_refused(dst, src):
    with pytest.raises(ValueError):
        precond._rearrange([(dst, src, 0, (1, 1, 4, 6), (0, 0, 6, 1), 6)])
    with pytest.raises(ValueError):  # also beside one that it can
        precond._rearrange([(torch.empty(1), torch.zeros(1), 0, (1,) * 4, (0,) * 4, 1),
                            (dst, src, 0, (1, 1, 4, 6), (0, 0, 6, 1), 6)])


@pytest.mark.gpu
def test_training_gradients_do_not_depend_on_it(default_dtype):
    print(f"[train] default {default_dtype}", flush=True)
    results = []
    for dtype in (torch.float32, default_dtype):
        torch.set_default_dtype(torch.float32)
        torch.manual_seed(1)
        net = precond.make_unet().cuda()
        x, y = torch.randn(2, 3, 40, 30).cuda(), 0.05 * torch.randn(2, 3, 40, 30).cuda()
        mask = torch.zeros(40, 30).cuda()
        mask[5:35, 4:26] = 1.0
        torch.set_default_dtype(dtype)
        loss, grads = precond.HipUNetTrainer(net).loss_and_grads(x, y, mask)
        results.append([loss] + [g for _, gw, gb in grads for g in (gw, gb)])
    for a, b in zip(*results):
        assert a.dtype == b.dtype == torch.float32 and torch.equal(a, b)
