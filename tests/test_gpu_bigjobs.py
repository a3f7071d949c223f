"""The int8 prompt kernels' BigJobs (moe_gate_up_big, moe_down_big) against the decode window calls on the same rows: the
same sums in the same order, so every output bit must agree.  Job sizes sit at the edges of the kernels' token groups (8),
tiles (16, 32) and of the few-row form (4, 8 rows); widths are every one the calls take, rows include part row tiles."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from sfnx_amd import moe
from sfnx_amd._abi import BIGJOB_INTS, JOB_INTS, PF_JOB

pytestmark = pytest.mark.gpu
TYPES = [orc.Q4_K, orc.Q5_K, orc.Q4_0, orc.Q5_1, orc.Q8_0]
SIZES = [1, 2, 3, 4, 5, 8, 9, 16, 17, 31, 32, 33, 48, 64]
WINDOW = 16


def store(wtype, n_mat, rows, cols, seed):
    x = torch.empty((n_mat * rows, cols), dtype=torch.float32, device="cuda")
    moe.synth_normal(x, seed, 0.02)
    g = torch.empty(n_mat * rows * moe.row_bytes(wtype, cols), dtype=torch.uint8, device="cuda")
    moe.quantize_weights(wtype, x, g)
    p = torch.empty_like(g)
    moe.store_pack(wtype, g, p, n_mat, rows, cols)
    return p


def jobs_of(sizes, rng, rows):
    """(BigJobs, windows of at most 16 rows of the same (expert, input row, output row) triples, pairs)"""
    P = sum(sizes)
    y, out = rng.integers(0, rows, P), rng.permutation(P)
    big = np.zeros((len(sizes), BIGJOB_INTS), np.int32)
    win = []
    at = 0
    for j, n in enumerate(sizes):
        big[j, 0], big[j, 1] = j % 3, n
        big[j, 2:2 + n], big[j, 2 + PF_JOB:2 + PF_JOB + n] = y[at:at + n], out[at:at + n]
        for k in range(0, n, WINDOW):
            m = min(WINDOW, n - k)
            w = np.zeros(JOB_INTS, np.int32)
            w[0], w[1] = j % 3, m
            w[2:2 + m], w[2 + WINDOW:2 + WINDOW + m] = y[at + k:at + k + m], out[at + k:at + k + m]
            win.append(w)
        at += n
    return torch.from_numpy(big).cuda(), torch.from_numpy(np.stack(win)).cuda(), P


@pytest.mark.parametrize("wtype", TYPES)
@pytest.mark.parametrize("n_in, n_out", [(512, 2048), (1024, 1056), (2048, 1024), (2560, 96), (4096, 160)])
@pytest.mark.parametrize("down, spare", [(False, 5), (True, 5), (True, 120), (True, 400), (True, 1200)])
def test_bigjobs_equal_windows(wtype, n_in, n_out, down, spare):
    """spare: job slots past the jobs, which the bound on their number counts: the more, the more row tiles (1 to 4) a block of
    down takes"""
    rng = np.random.default_rng(wtype + n_in)
    A = store(wtype, 3, n_out, n_in, 40 + wtype)
    sa = n_out * moe.row_bytes(wtype, n_in)
    rows = 40
    big, win, P = jobs_of(SIZES, rng, rows)
    nb = torch.tensor([big.shape[0], 0], dtype=torch.int32, device="cuda")
    nw = torch.tensor([win.shape[0], 0], dtype=torch.int32, device="cuda")
    cap = big.shape[0] + spare
    big = torch.cat([big, torch.zeros((spare, BIGJOB_INTS), dtype=torch.int32, device="cuda")])
    x = torch.from_numpy(rng.standard_normal((rows, 2 * n_in if down else n_in)).astype(np.float32)).cuda()
    got, want = (torch.full((P, n_out), 7.0, device="cuda") for _ in range(2))
    if down:
        moe.moe_down_big(A, sa, wtype, n_in, n_out, big, nb, cap, x, got)
        moe.moe_down(A, sa, wtype, n_in, n_out, win, nw, win.shape[0], WINDOW, x, want)
    else:
        xq = torch.empty(rows * (n_in // 32) * 36, dtype=torch.uint8, device="cuda")
        moe.quantize_q8_1(x, xq)
        moe.moe_gate_up_big(A, sa, wtype, n_in, n_out, big, nb, cap, xq, got)
        moe.moe_gate_up(A, sa, wtype, n_in, n_out, win, nw, win.shape[0], WINDOW, xq, want)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))


@pytest.mark.parametrize("wtype", [orc.Q4_K, orc.Q8_0])
def test_bigjobs_none(wtype):
    """no job at all writes nothing"""
    A = store(wtype, 1, 128, 512, 3)
    n0 = torch.zeros(2, dtype=torch.int32, device="cuda")
    jobs = torch.zeros((2, BIGJOB_INTS), dtype=torch.int32, device="cuda")
    out = torch.full((4, 128), 7.0, device="cuda")
    x = torch.zeros((4, 1024), device="cuda")
    moe.moe_down_big(A, 128 * moe.row_bytes(wtype, 512), wtype, 512, 128, jobs, n0, 2, x, out)
    assert torch.all(out == 7.0)


@pytest.mark.parametrize("wtype", TYPES)
@pytest.mark.parametrize("n_in, n_out", [(512, 32), (1024, 64), (2048, 32)])
def test_down_few_rows(wtype, n_in, n_out):
    """the fewest rows a store holds: one or two window blocks of two row tiles"""
    test_bigjobs_equal_windows(wtype, n_in, n_out, True, 5)


@pytest.mark.parametrize("wtype", [orc.Q4_0, orc.Q5_1, orc.Q8_0])
@pytest.mark.parametrize("n_in, n_out", [(512, 1056), (1024, 96), (2048, 2048)])
def test_down_row_tiles(wtype, n_in, n_out):
    """the window down call with one row tile a block and with two, which a larger bound on the job count selects: the
    same bits"""
    rng = np.random.default_rng(wtype + n_out)
    A = store(wtype, 3, n_out, n_in, 60 + wtype)
    _, win, P = jobs_of([1, 16, 7], rng, 20)
    nw = torch.tensor([win.shape[0], 0], dtype=torch.int32, device="cuda")
    x = torch.from_numpy(rng.standard_normal((20, 2 * n_in)).astype(np.float32)).cuda()
    out = []
    for cap in (win.shape[0], 4096):
        out.append(torch.full((P, n_out), 7.0, device="cuda"))
        moe.moe_down(A, n_out * moe.row_bytes(wtype, n_in), wtype, n_in, n_out, win, nw, cap, WINDOW, x, out[-1])
    torch.cuda.synchronize()
    assert torch.equal(out[0].view(torch.int32), out[1].view(torch.int32))
