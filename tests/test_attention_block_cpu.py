"""RoPE frequency tables of the attention block (``lagunalab_amd.attention.rope_frequencies``),
pinned by closed forms of the default and YaRN schedules (mlx-lm's ``initialize_rope`` is not in
this environment; the YaRN schedule follows the published method: frequencies of dims that
rotate more than ``beta_fast`` times over the original context are kept, those rotating fewer
than ``beta_slow`` times are divided by ``factor``, a linear ramp in between)."""
import math

import pytest
import torch

from lagunalab_amd.attention import rope_frequencies


def test_default_rope_is_theta_power():
    inv, dims, ms = rope_frequencies(128, {"rope_theta": 10000.0})
    assert dims == 128 and ms == 1.0 and inv.shape == (64,)
    assert torch.allclose(inv.double(), 10000.0 ** (-torch.arange(0, 128, 2).double() / 128))
    inv, dims, _ = rope_frequencies(128, {"rope_theta": 1e4, "partial_rotary_factor": 0.5})
    assert dims == 64 and inv.shape == (32,)
    assert inv[0] == 1.0 and inv[1].item() == pytest.approx(1e4 ** (-2 / 64), rel=1e-7)  # fp32


def test_yarn_limits_and_mscale():
    p = {"rope_type": "yarn", "rope_theta": 5e5, "factor": 32.0, "partial_rotary_factor": 0.5,
         "original_max_position_embeddings": 4096}
    inv, dims, ms = rope_frequencies(128, p)
    base, _, _ = rope_frequencies(128, {"rope_theta": 5e5, "partial_rotary_factor": 0.5})
    assert dims == 64
    assert ms == pytest.approx(0.1 * math.log(32.0) + 1.0)
    # correction range of the published method, in rotated-pair index
    cd = lambda r: dims * math.log(4096 / (r * 2 * math.pi)) / (2 * math.log(5e5))
    low, high = max(math.floor(cd(32)), 0), min(math.ceil(cd(1)), dims - 1)
    assert 0 < low < high < dims // 2
    assert torch.equal(inv[:low + 1], base[:low + 1])             # fast dims: unchanged
    assert torch.allclose(inv[high:], base[high:] / 32.0)         # slow dims: interpolated
    mid = (low + high) // 2
    t = (mid - low) / (high - low)
    assert inv[mid].item() == pytest.approx(base[mid].item() * ((1 - t) + t / 32.0), rel=1e-6)
    # factor 1: the default table, no scaling
    inv1, _, ms1 = rope_frequencies(128, dict(p, factor=1.0))
    assert torch.allclose(inv1, base) and ms1 == 1.0
    # mscale_all_dim equal to mscale cancels the attention factor
    _, _, ms2 = rope_frequencies(128, dict(p, mscale=0.7, mscale_all_dim=0.7))
    assert ms2 == pytest.approx(1.0)


def test_unknown_rope_type_rejected():
    with pytest.raises(ValueError, match="rope_type"):
        rope_frequencies(128, {"rope_type": "llama3", "rope_theta": 1e4})


def test_row_form_leaves_transforms_and_other_layouts_to_the_library():
    """linear() of 2 to 16 rows: off the GPU, under vmap or forward mode, with gradients wanted, in
    another type or layout, the library product is what runs."""
    import torch
    from torch.autograd import forward_ad
    from lagunalab_amd.attention import linear
    g = torch.Generator().manual_seed(1)
    x, w = torch.randn((4, 64), generator=g), torch.randn((24, 64), generator=g)
    want = x @ w.t()
    assert torch.equal(linear(x, w), want)
    assert torch.allclose(torch.vmap(lambda a: linear(a, w))(x.reshape(2, 2, 64)).reshape(4, 24), want)
    xg = x.clone().requires_grad_()
    linear(xg, w).sum().backward()
    assert torch.allclose(xg.grad, w.sum(0).expand(4, 64), atol=1e-4)
    with forward_ad.dual_level():
        d = linear(forward_ad.make_dual(x, torch.ones_like(x)), w)
        assert torch.allclose(forward_ad.unpack_dual(d).tangent, w.sum(1).expand(4, 24), atol=1e-4)
    assert torch.equal(linear(x, w.t().contiguous().t()), x @ w.t().contiguous())


def test_unwatched_calls_only_outside_tracing_modes_and_autocast():
    """The row form's launch is not seen by the dispatcher, so every context that works on what the
    dispatcher sees has to be told apart from a plain call."""
    import torch
    from torch.autograd import forward_ad
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.overrides import TorchFunctionMode
    from torch.utils.flop_counter import FlopCounterMode
    from lagunalab_amd.attention import _unwatched
    x, w = torch.randn((4, 8)), torch.randn((3, 8))
    seen = []

    def call(a, b=w):
        seen.append(_unwatched(a, b))
        return a @ b.t()

    class Mode(TorchFunctionMode):
        def __torch_function__(self, fn, types, args=(), kwargs=None):
            return fn(*args, **(kwargs or {}))

    call(x)
    with torch.inference_mode():
        call(x)
    with torch.device("cpu"):
        call(x)
    assert seen == [True] * 3
    seen.clear()
    torch.jit.trace(call, (x,), check_trace=False)
    make_fx(lambda a, b: call(a, b))(x, w)
    make_fx(lambda a, b: call(a, b), tracing_mode="fake")(x, w)
    with FlopCounterMode(display=False):
        call(x)
    with torch.autocast("cpu", dtype=torch.bfloat16):
        call(x)
    with Mode():
        call(x)
    torch.vmap(call)(x)
    call(x.clone().requires_grad_())
    call(torch.nn.Parameter(x))
    with forward_ad.dual_level():
        call(forward_ad.make_dual(x, x))
    assert len(seen) >= 10 and not any(seen)


@pytest.mark.parametrize("rows,N,K,pays", [
    (2, 1023, 2048, 0), (2, 1024, 1023, 0), (16, 1024, 1024, 1), (16, 4096, 2048, 1), (16, 2048, 2049, 0),
    (16, 2048, 3072, 1), (16, 4096, 4096, 1), (2, 2048, 4097, 0), (2, 4097, 3072, 0), (12, 4097, 1536, 1),
    (13, 8192, 2048, 0), (4, 8192, 1535, 1), (5, 8192, 1535, 0), (8, 8193, 1793, 1), (8, 8193, 1792, 0),
    (9, 8193, 2048, 0), (8, 12289, 2048, 0)])
def test_row_form_only_where_it_was_measured_faster(rows, N, K, pays):
    from lagunalab_amd.attention import _row_form_pays
    assert _row_form_pays(rows, N, K) == bool(pays)


def test_linear_refuses_rows_of_no_inputs():
    import torch
    from lagunalab_amd.attention import linear
    with pytest.raises(ValueError):
        linear(torch.empty((3, 0), dtype=torch.bfloat16), torch.empty((4, 0), dtype=torch.bfloat16))
