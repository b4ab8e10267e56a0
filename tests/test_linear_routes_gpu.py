"""Which calls of `ops.linear` and of the small projection kernels reach a kernel: those the library's F.linear would refuse stay
refused, and those it serves in a way a kernel cannot (broadcast bias, vmap, forward mode) stay with it."""
import pytest
import torch
import torch.nn.functional as F
from torch.autograd import forward_ad

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _r(*s, dtype=torch.float32):
    return torch.randn(*s, generator=torch.Generator().manual_seed(len(s) + s[-1])).to(DEV, dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_mismatched_operands_are_refused(dtype):
    from native_sparse_attention_pytorch_amd import ops
    x, fn = _r(8, 64, dtype=dtype), (ops.linear_f32 if dtype == torch.float32 else ops.skinny_linear)
    other = torch.bfloat16 if dtype == torch.float32 else torch.float32
    supported = ops.linear_f32_supported if dtype == torch.float32 else ops.skinny_linear_supported
    for w, b in ((_r(16, 32, dtype=dtype), None), (_r(16, 128, dtype=dtype), None), (_r(16, 64, dtype=dtype), _r(8, dtype=dtype)),
                 (_r(16, 64, dtype=dtype), _r(16, dtype=other))):
        assert w.shape[1] == 64 or not supported(x, w)
        with pytest.raises(RuntimeError):
            fn(x, w, b)
        with torch.no_grad(), pytest.raises(RuntimeError):
            ops.linear(x, w, b)


@torch.no_grad()
def test_what_only_the_operator_serves():
    from native_sparse_attention_pytorch_amd import ops
    x, w = _r(8, 64), _r(16, 64)
    one = _r(1)
    # fp32 sums of 64 products in another order: 64 x 2^-24 of the magnitudes (at most ~ 64 x 16)
    close = lambda a, b: torch.testing.assert_close(a, b, rtol=0, atol=64 * 2 ** -24 * 1024)
    close(ops.linear(x, w, one), F.linear(x, w) + one)
    close(torch.vmap(lambda t: ops.linear(t, w))(x[:, None]), F.linear(x[:, None], w))
    with forward_ad.dual_level():
        y = ops.linear(forward_ad.make_dual(x, x + 1), w)
        close(forward_ad.unpack_dual(y).tangent, F.linear(x + 1, w))
    # the weight batched: an address would be that of the whole stack
    stack = _r(3, 16, 64)
    close(torch.vmap(lambda u: ops.linear(x, u))(stack), F.linear(x, stack.reshape(48, 64)).view(8, 3, 16).transpose(0, 1))


@torch.no_grad()
@pytest.mark.parametrize("trace", ["compile", "make_fx", "make_fx fake", "make_fx pre_dispatch", "jit.trace"])
def test_traces_record_the_operator(trace):
    """A traced projection computes on the inputs it is run on: a kernel launched while tracing would leave its result as a constant."""
    from torch.fx.experimental.proxy_tensor import make_fx
    from native_sparse_attention_pytorch_amd import ops
    x, w, b = _r(8, 64), _r(16, 64), _r(16)
    args, other = (x, w, b), (x.flip(0) * 2, w + 1, b)
    if trace == "compile":
        torch._dynamo.reset()
        run = torch.compile(ops.linear, backend="eager", fullgraph=True)
        run(*args)
    elif trace == "jit.trace":
        run = torch.jit.trace(ops.linear, args, check_trace=False)
    else:
        run = make_fx(ops.linear, tracing_mode="fake" if "fake" in trace else "real", pre_dispatch="pre" in trace)(*args)
    got, want = run(*other), F.linear(*other)
    torch.testing.assert_close(got, want, rtol=0, atol=64 * 2 ** -24 * 1024)
