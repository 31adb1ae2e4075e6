"""Which calls of `linear` may pass torch's dispatcher by: those that nothing else looks at."""
import pytest
import torch
import torch.autograd.forward_ad as fwd
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode

from zipage_amd.layers import linear
from zipage_amd.layers.linear import ResidualLinear, _seen_by_others


class _Sub(torch.Tensor):
    pass


class _Mode(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def _under_vmap(x, w, look):
    torch.func.vmap(lambda a: (look(a, w), a)[1])(x.expand(2, -1, -1))


def _under_jvp(x, w, look):
    torch.func.jvp(lambda a: (look(a, w), a)[1], (x,), (x,))


def _under_dual(x, w, look):
    with fwd.dual_level():
        look(fwd.make_dual(x, x), w)


def _under_grad(x, w, look):
    look(x, w.clone().requires_grad_())


def _under_autocast(x, w, look):
    torch.set_autocast_enabled("cuda", True)                  # torch.autocast asks for a device that is there
    try:
        look(x, w)
    finally:
        torch.set_autocast_enabled("cuda", False)


def _under_fx(x, w, look):
    make_fx(lambda a: (look(a, w), a + 1)[1])(x)


def _under_jit(x, w, look):
    torch.jit.trace(lambda a: (look(a, w), a + 1)[1], x, check_trace=False)


def _under_fake(x, w, look):
    with FakeTensorMode() as m:
        look(m.from_tensor(x), m.from_tensor(w))


def _as_subclass(x, w, look):
    look(x.as_subclass(_Sub), w)


def _under_mode(x, w, look):
    with _Mode():
        look(x, w)


@pytest.mark.filterwarnings("ignore")
@pytest.mark.parametrize("under", [_under_vmap, _under_jvp, _under_dual, _under_grad, _under_autocast, _under_fx, _under_jit, _under_fake, _as_subclass,
                                   _under_mode])
def test_calls_that_others_look_at(under):
    x, w, seen = torch.randn(5, 64), torch.randn(96, 64), []
    under(x, w, lambda a, b: seen.append(_seen_by_others(a, b)))
    assert seen == [True]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_device_tensors_without_storage(dtype):
    with FakeTensorMode():
        x, w = torch.empty(5, 64, dtype=dtype, device="cuda"), torch.empty(96, 64, dtype=dtype, device="cuda")
        assert linear(x, w).shape == (5, 96)
        assert ResidualLinear(w).forward(x).shape == (1, 5, 96)


# on either side of the lines that measuring drew, with weights from memory
@pytest.mark.parametrize("n,k,m,few", [(1, 1024, 4096, True), (16, 4096, 4096, True), (8, 12288, 4096, True), (8, 12288, 1024, False), (8, 12288, 9216, False),
                                       (8, 8192, 4096, False), (16, 128, 32768, False), (16, 256, 32768, True), (8, 1024, 65536, False),
                                       (8, 2048, 151936, True), (17, 4096, 4096, True), (17, 4096, 6144, False), (32, 4096, 24576, False),
                                       (24, 1024, 16384, True), (24, 1024, 20480, False), (24, 2048, 8192, True), (24, 2048, 9216, False),
                                       (32, 64, 5120, False), (48, 1024, 4096, True), (48, 3072, 1024, True), (48, 3072, 2048, False),
                                       (48, 3072, 256, False), (48, 64, 8192, False), (64, 1024, 16384, False), (65, 1024, 1024, False),
                                       (0, 64, 64, False), (4, 48, 64, False), (4, 64, 66, False)])
def test_which_sizes_are_few_rows(n, k, m, few):
    from zipage_amd.layers.linear import _few_rows
    assert _few_rows(n, k, m) == few


@pytest.mark.parametrize("n,k,m,tiles", [(64, 1024, 1024, False), (65, 1024, 1024, True), (256, 1024, 1024, True), (257, 1024, 1024, False),
                                         (65, 64, 1024, False), (65, 96, 1024, True), (128, 1024, 8192, True), (128, 1024, 8196, False),
                                         (129, 1024, 5440, True), (129, 1024, 5444, False), (256, 1024, 4096, True), (256, 1056, 4096, False),
                                         (256, 1056, 2048, True), (128, 2048, 8192, True), (128, 2080, 4096, True), (128, 2080, 4128, False),
                                         (96, 2080, 4096, False), (129, 2080, 1024, False), (112, 4096, 4096, False), (113, 4096, 4096, True),
                                         (128, 4128, 1024, False), (100, 48, 64, False), (100, 128, 66, False), (100, 144, 64, False)])
def test_which_sizes_are_row_tiles(n, k, m, tiles):
    from zipage_amd.layers.linear import _few_rows, _row_tiles
    assert _row_tiles(n, k, m) == tiles and not (_row_tiles(n, k, m) and _few_rows(n, k, m))


# each line of the rule from both sides
@pytest.mark.parametrize("n,k,m,split", [(16, 12288, 4096, False), (17, 12288, 4096, True), (32, 4608, 4096, False), (32, 12288, 4868, False),
                                         (32, 8192, 1980, False), (24, 4096, 24576, True), (24, 4096, 151936, True), (24, 992, 151936, False),
                                         (64, 1024, 151936, True), (65, 1024, 151936, False), (112, 4096, 151936, True), (113, 4096, 151936, False),
                                         (33, 4096, 6144, True), (33, 4096, 10244, False), (48, 3072, 1024, True), (48, 3072, 2048, False),
                                         (48, 2528, 1024, False), (64, 8192, 1024, False), (64, 8224, 1024, True), (65, 4096, 4096, False),
                                         (89, 4096, 4096, True), (65, 4096, 6144, True), (128, 12288, 1020, False), (128, 4096, 24576, True),
                                         (129, 4096, 24576, False), (129, 4096, 6144, True), (192, 4096, 4096, True), (193, 4096, 4096, False),
                                         (256, 4096, 6144, True), (256, 12288, 4096, True), (257, 12288, 4096, False), (256, 4064, 6144, False),
                                         (128, 4096, 32768, True), (129, 4096, 32768, False), (24, 2048, 26880, True), (64, 2016, 32768, False),
                                         (64, 4096, 26876, False), (64, 4096, 32772, False), (255, 4096, 6144, False), (224, 4096, 6144, True), (100, 6160, 4096, False), (100, 6144, 4098, False)])
def test_which_sizes_are_split(n, k, m, split):
    from zipage_amd.layers.linear import _split_rows
    assert _split_rows(n, k, m) == split


@pytest.mark.parametrize("n", [0, 1, 16, 17, 32, 64, 65, 128, 256])
@pytest.mark.parametrize("k,m", [(1024, 0), (4096, 0), (0, 1024), (0, 0)])
def test_products_of_nothing_stay_with_the_library(n, k, m):
    from zipage_amd.layers.linear import _few_rows, _row_tiles, _split_rows
    assert not (_few_rows(n, k, m) or _row_tiles(n, k, m) or _split_rows(n, k, m))


# where either kernel was slower than the library: from both sides of the lines that keep these sizes there
@pytest.mark.parametrize("n,k,m,tiles", [(65, 288, 8192, False), (65, 320, 8192, True), (65, 288, 4096, True), (69, 2016, 7620, True), (69, 2048, 7620, False),
                                         (69, 2048, 4096, True), (112, 2048, 4100, False), (113, 2048, 4100, True), (129, 288, 4096, False),
                                         (120, 4096, 1024, True), (120, 4096, 1028, False), (120, 4064, 1776, True), (128, 4096, 2176, False),
                                         (128, 4096, 2180, True), (127, 4096, 3964, False), (127, 4096, 3968, True)])
def test_which_sizes_are_no_row_tiles(n, k, m, tiles):
    from zipage_amd.layers.linear import _row_tiles
    assert _row_tiles(n, k, m) == tiles


@pytest.mark.parametrize("n,k,m,split", [(48, 8192, 29952, True), (48, 8224, 29952, False), (49, 4608, 29952, True), (49, 4640, 29952, False),
                                         (128, 4608, 32256, True), (128, 4640, 32256, False), (32, 5120, 24576, True), (32, 5152, 24576, False),
                                         (128, 8192, 24576, True), (128, 8224, 24576, False), (32, 5120, 120000, True), (33, 5088, 120000, True),
                                         (33, 5120, 120000, False), (80, 4096, 151936, False), (81, 4096, 151936, True), (96, 4096, 140000, True),
                                         (97, 4096, 140000, False), (97, 4096, 147456, True), (144, 5888, 1788, False), (144, 5888, 1792, True),
                                         (144, 6656, 1280, True), (80, 8192, 1660, False), (80, 8192, 1664, True), (81, 8192, 1280, True), (80, 8224, 1280, True)])
def test_which_sizes_stay_whole(n, k, m, split):
    from zipage_amd.layers.linear import _split_rows
    assert _split_rows(n, k, m) == split
