"""Continuous batching in one library call: up to 16 int8 rows read where they
lie, other batches gathered first; requests off a 16-byte boundary, K that
fills no step or no fragment, more requests than one gather launch takes,
packed weights.  Outputs are each request's exact product, the staging buffer
holds the concatenation, and the workspace serves the next call."""
import pytest
import torch

from oracle import rns_oracle as ro

pytestmark = pytest.mark.gpu

DENSE4 = (255, 253, 251, 247)
DENSE6 = DENSE4 + (241, 239)


def exact(a, w_nk):
    return torch.from_numpy(ro.exact_matmul(a.cpu().numpy(), w_nk.t().numpy()))


@pytest.mark.parametrize("rows", [(1,), (1, 1, 1, 1), (3, 1, 12), (16,), (8, 9), (5, 40, 1), (1,) * 35, (2,) * 8])
@pytest.mark.parametrize("k,n", [(768, 100), (80, 17), (777, 64), (4096, 48), (1040, 7)])
@pytest.mark.parametrize("dtype,packed", [(torch.int8, False), (torch.int16, False), (torch.int16, True), (torch.int32, False)])
def test_merged_products(backend, rows, k, n, dtype, packed):
    gen = torch.Generator().manual_seed(sum(rows) + k)
    lim = 127 if dtype == torch.int8 else 2047
    moduli = DENSE4 if dtype == torch.int8 else DENSE6
    w = torch.randint(-lim, lim + 1, (n, k), generator=gen, dtype=torch.int32).to(torch.int8 if lim == 127 else torch.int16)
    prepared = (backend.prepare_weight_packed_nk if packed else backend.prepare_weight_nk)(w.cuda(), moduli)
    ws = backend.create_request_batch_workspace(device=torch.device("cuda"), dtype=dtype, rows_per_request=rows, k=k,
                                                channels=len(moduli), n=n)
    for shift in (0, 1):  # the second time every request starts off a 16-byte boundary
        requests = []
        for r in rows:
            t = torch.empty((r * k + shift,), dtype=dtype, device="cuda")[shift:].view(r, k)
            requests.append(t.copy_(torch.randint(-lim - 1, lim + 1, (r, k), generator=gen, dtype=torch.int32)))
        backend.reset_stats()
        outs = backend.matmul_prepared_fused_requests(requests, prepared, workspace=ws)
        assert backend.stats_snapshot() == {
            "encode_centered_calls": 1, "encode_centered_values": sum(rows) * k, "fused_gemm_calls": 1,
            f"fused_gemm_channels_{len(moduli)}": 1, "continuous_batch_calls": 1, "continuous_batch_requests": len(rows)}
        assert torch.equal(ws.activations, torch.cat(requests))
        assert len(outs) == len(rows) and outs[0].data_ptr() == ws.fused.output.data_ptr()
        for request, out in zip(requests, outs):
            assert torch.equal(out.cpu(), exact(request, w))
    clones = backend.matmul_prepared_fused_requests(requests, prepared, clone_outputs=True)
    assert torch.equal(torch.cat(clones), ws.fused.output)


# a long K and few columns, on both sides of where the rows are gathered first
# and the product splits K over workgroups
@pytest.mark.parametrize("rows,k,n", [((5, 6), 8192, 100), ((5, 7), 8192, 100), ((16,), 5632, 300), ((16,), 5648, 300),
                                      ((1, 3), 12288, 40), ((16,), 3072, 40)])
def test_long_k(backend, rows, k, n):
    gen = torch.Generator().manual_seed(k)
    w = torch.randint(-127, 128, (n, k), generator=gen, dtype=torch.int32).to(torch.int8)
    prepared = backend.prepare_weight_nk(w.cuda(), DENSE4)
    ws = backend.create_request_batch_workspace(device=torch.device("cuda"), dtype=torch.int8, rows_per_request=rows, k=k,
                                                channels=4, n=n)
    for _ in range(2):
        requests = [torch.randint(-128, 128, (r, k), generator=gen, dtype=torch.int32).to(torch.int8).cuda() for r in rows]
        outs = backend.matmul_prepared_fused_requests(requests, prepared, workspace=ws)
        assert torch.equal(ws.activations, torch.cat(requests))
        for request, out in zip(requests, outs):
            assert torch.equal(out.cpu(), exact(request, w))


def test_refusals(backend):
    w = torch.ones((16, 64), dtype=torch.int8).cuda()
    prepared = backend.prepare_weight_nk(w, DENSE4)
    x = torch.ones((2, 64), dtype=torch.int8).cuda()
    ws = backend.create_request_batch_workspace(device=x.device, dtype=torch.int8, rows_per_request=(2,), k=64,
                                                channels=4, n=16)
    for requests, kw in (([], {}), ([x, x.to(torch.int16)], {}), ([x[:, :32].contiguous()], {}), ([x.t()], {}), ([x, x], {"workspace": ws}),
                         ([x], {"lut_channels": 3}), ([x.float()], {}), ([x.cpu()], {})):
        with pytest.raises(ValueError):
            backend.matmul_prepared_fused_requests(requests, prepared, **kw)


@pytest.mark.parametrize("rows", [(2, 2), (20, 20)])
def test_requests_inside_the_staging_buffer_are_refused(backend, rows):
    """Rows that would be copied over each other: refused, whatever their number."""
    prepared = backend.prepare_weight_nk(torch.ones((16, 64), dtype=torch.int8).cuda(), DENSE4)
    ws = backend.create_request_batch_workspace(device=torch.device("cuda"), dtype=torch.int8, rows_per_request=rows,
                                                k=64, channels=4, n=16)
    ws.activations.fill_(1)
    half = rows[0]
    with pytest.raises(RuntimeError):
        backend.matmul_prepared_fused_requests([ws.activations[half:], ws.activations[:half]], prepared, workspace=ws)


@pytest.mark.parametrize("rows", [(1, 1), (4, 12), (20, 20)])
def test_outputs_over_a_request(backend, rows):
    """Outputs written where a request lies, or begin inside it."""
    k, n = 512, 64
    gen = torch.Generator().manual_seed(sum(rows))
    w = torch.randint(-127, 128, (n, k), generator=gen, dtype=torch.int32).to(torch.int8)
    prepared = backend.prepare_weight_nk(w.cuda(), DENSE4)
    ws = backend.create_request_batch_workspace(device=torch.device("cuda"), dtype=torch.int8, rows_per_request=rows, k=k,
                                                channels=4, n=n)
    m, given = sum(rows), [torch.randint(-128, 128, (r, k), generator=gen, dtype=torch.int32).to(torch.int8) for r in rows]
    buffer = torch.empty((2 * m * (k + 8 * n),), dtype=torch.int8, device="cuda")
    for lo in (0, k // 2):
        ws.fused.output = buffer[lo:lo + 8 * m * n].view(torch.int64).view(m, n)
        for _ in range(5):
            requests, at = [], 0
            for r, x in zip(rows, given):
                requests.append(buffer[at:at + r * k].view(r, k).copy_(x))
                at += r * k
            outs = backend.matmul_prepared_fused_requests(requests, prepared, workspace=ws)
            for x, out in zip(given, outs):
                assert torch.equal(out.cpu(), exact(x, w))


def test_a_request_without_rows(backend):
    """A batch workspace put together by hand may hold a request of no rows."""
    from rns_llm_amd.backends.hip_backend import RNSRequestBatchWorkspace

    gen = torch.Generator().manual_seed(2)
    w, x = (torch.randint(-127, 128, shape, generator=gen, dtype=torch.int32).to(torch.int8) for shape in ((16, 64), (3, 64)))
    prepared, dev = backend.prepare_weight_nk(w.cuda(), DENSE4), torch.device("cuda")
    ws = RNSRequestBatchWorkspace(activations=torch.empty((3, 64), dtype=torch.int8, device=dev),
                                  fused=backend.create_workspace(device=dev, channels=4, m=3, n=16, k=64),
                                  rows_per_request=(1, 0, 2), k=64)
    rows = x.cuda()
    outs = backend.matmul_prepared_fused_requests([rows[:1], rows[1:1], rows[1:]], prepared, workspace=ws)
    assert [o.shape[0] for o in outs] == [1, 0, 2]
    assert torch.equal(torch.cat(outs).cpu(), exact(x, w))
