"""RNSLinear on a few rows: quantized inside the product, one launch.  Every
float type, rows and widths at the edges of the rule (16 rows, 8192 values, K
that fills no K step, no vector or no fragment, N past a column block), and
non-finite inputs, against the CPU float chain and the quantizer's own
kernels (an adaptive layer takes those)."""
import pytest
import torch

from oracle import linear_oracle
from rns_llm_amd import RNSLinear

pytestmark = pytest.mark.gpu


def layer_of(backend, k, n, dtype, bias=True, **kw):
    torch.manual_seed(k + n)
    return RNSLinear(k, n, bias=bias, mode="rns", backend=backend, **kw).to(device="cuda", dtype=dtype).eval()


@pytest.mark.parametrize("rows,k,n", [(1, 768, 2304), (1, 8192, 48), (2, 4096, 33), (16, 512, 17), (16, 513, 64), (10, 777, 40),
                                      (13, 600, 31), (3, 1001, 70), (1, 515, 16), (8, 1024, 100), (17, 481, 32), (9, 911, 16),
                                      # both sides of the lines where the quantizer's own kernels take over
                                      (4, 768, 8192), (4, 768, 8193), (4, 1024, 97), (4, 1025, 97), (5, 777, 97)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bias", [True, False])
def test_rows_equal_the_float_chain(backend, rows, k, n, dtype, bias):
    layer = layer_of(backend, k, n, dtype, bias)
    gen = torch.Generator().manual_seed(rows)
    x = torch.randn((rows, k), generator=gen).to(dtype)
    x[-1, -1] = 7.5  # the largest value at the very end
    with torch.no_grad():
        y = layer(x.cuda())
        # rows that start off a 16-byte boundary
        shifted = torch.empty((rows * k + 1,), dtype=dtype, device="cuda")[1:].view(rows, k)
        shifted.copy_(x)
        assert torch.equal(layer(shifted), y)
    want, _ = linear_oracle.linear_forward(x, layer.weight.detach().cpu(),
                                           layer.bias.detach().cpu() if bias else None, bits=8)
    assert torch.equal(y.cpu(), want)


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -float("inf")])
def test_non_finite_inputs(backend, bad):
    """As the quantizer's kernels: 17 rows take those."""
    layer = layer_of(backend, 512, 64, torch.float32)
    x = torch.randn((17, 512), generator=torch.Generator().manual_seed(1))
    x[0, 3] = bad
    with torch.no_grad():
        few, many = layer(x[:1].cuda()), layer(x.cuda())[:1]
    assert torch.equal(few.isnan(), many.isnan()) and few.isnan().any()
    assert torch.equal(few.nan_to_num(0.0), many.nan_to_num(0.0))


def test_zero_input_and_replays(backend):
    layer = layer_of(backend, 768, 200, torch.float16)
    x = torch.zeros((2, 768), dtype=torch.float16, device="cuda")
    with torch.no_grad():
        assert torch.equal(layer(x), layer.bias.expand(2, -1))
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            layer(x)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            y = layer(x)
        for seed in range(3):
            x.copy_(torch.randn((2, 768), generator=torch.Generator().manual_seed(seed)))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, layer(x))


@pytest.mark.parametrize("shift", [0, -256, 512])
@pytest.mark.parametrize("rows,k,n", [(1, 768, 768), (4, 1024, 1024), (3, 512, 1000)])
def test_outputs_over_the_activations(backend, rows, k, n, shift):
    """The library call with out_dev inside x_dev: as into another buffer."""
    layer = layer_of(backend, k, n, torch.float16)
    x = torch.randn((rows, k), generator=torch.Generator().manual_seed(n)).to(device="cuda", dtype=torch.float16)
    with torch.no_grad():
        want = layer(x)
        call = layer._bind_linear()
        buffer = torch.zeros((rows * max(k, n) + 2048,), dtype=torch.float16, device="cuda")
        scratch = backend.create_linear_scratch(call, rows, x.device)
        for _ in range(5):
            inside = buffer[1024:1024 + rows * k].view(rows, k).copy_(x)
            out = buffer[1024 + shift:1024 + shift + rows * n].view(rows, n)
            call(inside, rows, out, scratch)
            assert torch.equal(out, want)
