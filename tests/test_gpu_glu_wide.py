"""GPU: gated activations of prompts, four columns per thread where the rows are 16-byte aligned, against the same call on rows
that are not, which takes one column per thread: the arithmetic is the same, so the results are, bit for bit. test_gpu_epilogue
holds the one-column kernel to the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act,lanes", [(1, 0), (1, 16), (2, 0), (2, 8)])
@pytest.mark.parametrize("rows,cols,ldg,ldu", [(512, 2048, 2048, 2048),      # the smallest product that qualifies
                                               (373, 2883, 2884, 2888),      # a last piece of three columns
                                               (1048577, 1, 4, 4), (1, 1048578, 1048580, 1048580), (700, 2877, 5760, 5764)])
def test_glu_four_columns(hip, act, lanes, rows, cols, ldg, ldu):
    import torch
    print(f"glu act={act} lanes={lanes} rows={rows} cols={cols}", flush=True)
    gen = torch.Generator().manual_seed(rows + cols)
    g = torch.randn((rows, ldg), generator=gen) * 6
    u = torch.randn((rows, ldu), generator=gen) * 6
    edge = torch.tensor([7.0, 7.0001, -7.0, 40.0, -40.0, 0.0, -0.0, 1e-30, float("nan"), float("inf"), -float("inf")])
    g.view(-1)[:edge.numel()] = edge
    got = []
    for shift in (0, 1):   # floats off a 16-byte boundary
        gd = torch.zeros(rows * ldg + 4, device="cuda")
        ud = torch.zeros(rows * ldu + 4, device="cuda")
        gd[shift:shift + rows * ldg] = g.view(-1).cuda()
        ud[shift:shift + rows * ldu] = u.view(-1).cuda()
        torch.cuda.synchronize()
        args = (act, gd.data_ptr() + 4 * shift, ldg, ud.data_ptr() + 4 * shift, ldu, rows, cols)
        status = hip.glu_device_vector(*args, lanes) if lanes else hip.glu_device(*args)
        assert status == 0, hip.last_error()
        hip.synchronize()
        got.append(gd[shift:shift + rows * ldg].cpu().numpy().view(np.uint32).reshape(rows, ldg))
    nan = (got[0] & 0x7fffffff) > 0x7f800000
    assert np.array_equal(nan, (got[1] & 0x7fffffff) > 0x7f800000)
    assert np.array_equal(got[0][~nan], got[1][~nan])
    assert np.array_equal(got[0][:, cols:], g.numpy().view(np.uint32)[:, cols:])   # gap untouched
