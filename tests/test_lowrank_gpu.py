"""lowrank (eggroll.py:56-58) at the edges of its kernels: tile remainders of rows, outputs and contraction, the
one-launch form for few outputs, the tile sizes' rule, and the strides, dtypes and alignments the operands pass
reads. Against the formula in fp32 on bf16 operands; a product's or dot's bf16 rounding may go the other way where two
fp32 sums straddle a boundary, so the bound is one bf16 ulp of each plus the sums' order error (2^-20 of the terms)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device('cuda', 0)


def check(x, w, a, b, sign, div, got=None):
    from noise_amd.eggroll import lowrank
    m = x.shape[0]
    got = lowrank(x, w, a, b, sign, dir_div=div) if got is None else got
    bf = lambda t: t.bfloat16().float()
    d = torch.arange(m, device=DEV) // div
    xr, wr, br, ar = bf(x), bf(w), bf(b)[d], a.float()[d]
    prod = torch.stack([xr[i] @ wr.t() for i in range(m)])
    dot = (xr * br[:, None, :]).sum(-1, keepdim=True)
    s = sign[:, None, None]
    ref = bf(prod) + s * bf(dot) * ar[:, None, :]
    size = torch.stack([xr[i].abs() @ wr.abs().t() for i in range(m)])
    dsize = (xr * br[:, None, :]).abs().sum(-1, keepdim=True)
    bound = (prod.abs() * 2.0 ** -7 + size * 2.0 ** -20
             + (s * ar[:, None, :]).abs() * (dot.abs() * 2.0 ** -7 + dsize * 2.0 ** -20) + 1e-30)
    assert got.shape == ref.shape and got.dtype == torch.float32
    assert ((got - ref).abs() <= bound).all()


def inputs(m, T, n_in, n_out, div, dtype, seed):
    g = torch.Generator(DEV).manual_seed(seed)
    r = lambda *s: torch.randn(*s, device=DEV, generator=g)
    dirs = -(-m // div)
    return r(m, T, n_in).to(dtype), r(n_out, n_in) * 0.2, r(dirs, n_out), r(dirs, n_in), r(m) * 0.3


@pytest.mark.parametrize('m,T,n_in,n_out', [
    (1, 1, 1, 1), (3, 5, 33, 7), (2, 33, 256, 16), (2, 17, 257, 16), (5, 51, 64, 17), (1, 127, 65, 20),
    (1, 128, 63, 128), (3, 43, 512, 129), (2, 129, 192, 260), (4, 256, 512, 256), (9, 911, 128, 2049),
    (16, 256, 320, 4096)])
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
def test_lowrank_edges(m, T, n_in, n_out, dtype):
    print(m, T, n_in, n_out, dtype, flush=True)
    x, w, a, b, sign = inputs(m, T, n_in, n_out, 2, dtype, m + T)
    check(x, w, a, b, sign, 2)
    check(x, w.bfloat16(), a, b, sign, 2)
    check(x[:1].expand(m, T, n_in), w, a, b, sign, 2)  # shared over the members


def test_lowrank_views():
    x, w, a, b, sign = inputs(6, 40, 512, 96, 1, torch.float32, 3)
    bf = x.bfloat16()
    wide = torch.randn(6, 40, 1031, device=DEV)
    cases = dict(columns=x[..., 64:192], odd_columns=wide[..., 3:131], every_other=bf[:, ::2], transposed=bf.transpose(0, 1),
                 inner=x.transpose(1, 2), tokens_expanded=bf[:, :1].expand(6, 40, 512), misaligned=wide.bfloat16()[..., 1:513],
                 members_reversed=bf.flip(0)[::2], half=x.half())
    for name, v in cases.items():
        print(name, tuple(v.shape), v.stride(), flush=True)
        m, T, n_in = v.shape
        for div in (1, 3):
            s = torch.randn(m, device=DEV) * 0.3
            aa, bb = torch.randn(m, 96, device=DEV), torch.randn(m, n_in, device=DEV)
            check(v, torch.randn(96, n_in, device=DEV) * 0.2, aa, bb, s, div)
    rows = torch.randn(6, 96 + 512 + 3, device=DEV)
    check(x, w, rows[:, :96], rows[:, 96:608], sign, 1)        # noise as column views of one table
    check(x, w, rows[:, 1:97], rows[:, 98:610], sign, 1)       # off the 16 B alignment
    check(x[:1].expand(6, 40, 512), w, rows[:, 1:97], rows[:, 98:610], sign, 1)
    check(x, w.t().contiguous().t(), a.bfloat16(), b.half(), sign, 1)
    check(x.transpose(1, 2)[:1].expand(6, 512, 40), torch.randn(18, 40, device=DEV), torch.randn(6, 18, device=DEV),
          torch.randn(6, 40, device=DEV), sign, 1)             # shared, no unit inner stride, outputs off the groups of 4


@pytest.mark.parametrize('m,T,n_in,n_out,div', [(1301, 2, 320, 20, 1), (1301, 5, 512, 4, 2), (1027, 3, 64, 1040, 3), (9, 1, 300, 8, 2),
                                                (2049, 129, 128, 32, 2)])
def test_shared_rows_of_few_tokens(m, T, n_in, n_out, div):
    """Few token tiles: the expansion's directions are shared out over workgroups, the last of them with fewer."""
    x, w, a, b, sign = inputs(m, T, n_in, n_out, div, torch.bfloat16, m + T)
    check(x[:1].expand(m, T, n_in), w, a, b, sign, div)


def test_shared_rows_of_few_tokens_take_no_longer_than_copies():
    """4,000 members on two shared rows: one workgroup that walks all of them took 20 times the call on copied rows."""
    from noise_amd.eggroll import lowrank
    x, w, a, b, sign = inputs(4000, 2, 1024, 16, 2, torch.bfloat16, 1)

    def ms(v):
        times = []
        for _ in range(7):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(20):
                lowrank(v, w, a, b, sign, dir_div=2)
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end))
        return sorted(times)[3]

    assert ms(x[:1].expand(4000, 2, 1024)) <= 4 * ms(x)


@pytest.mark.parametrize('m,n_in,n_out', [(65537, 32, 18), (2 ** 19 + 1, 32, 1), (2 ** 19 + 1, 8, 7)])
def test_more_rows_than_one_launch_has_waves(m, n_in, n_out):
    """1024 rows per member, past 2^26 rows for the operands' wave per row and 2^29 for the narrow form's eight lanes per row:
    a launch has fewer than 2^32 threads. A member's rows are one row repeated, so its outputs are that row's."""
    from noise_amd.eggroll import lowrank
    print(m, n_in, n_out, flush=True)
    x, w, a, b, sign = inputs(m, 1, n_in, n_out, 2, torch.bfloat16, n_out)
    few = lowrank(x, w, a, b, sign, dir_div=2)
    got = lowrank(x.expand(m, 1024, n_in), w, a, b, sign, dir_div=2)
    assert torch.equal(got[:, 0], few[:, 0]) and torch.equal(got.amin(1), few[:, 0]) and torch.equal(got.amax(1), few[:, 0])


@pytest.mark.parametrize('n_in,n_out', [(512, 18), (1024, 1), (64, 131)])
def test_shared_rows_are_not_copied_per_member(n_in, n_out):
    """x broadcast over the members: the scratch memory stays within the outputs' size in whole groups of 4 twice over, and
    the shared rows' and weights' own."""
    from noise_amd.eggroll import lowrank
    m, T = 256, 1024
    x, w, a, b, sign = inputs(1, T, n_in, n_out, 1, torch.bfloat16, 5)
    a, b, sign = (torch.randn(m, n, device=DEV) for n in (n_out, n_in, 1))
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    got = lowrank(x.expand(m, T, n_in), w, a, b, sign[:, 0], dir_div=1)
    used = torch.cuda.max_memory_allocated() - before
    assert used <= 8 * m * T * -(-n_out // 4) * 4 + 16 * T * (n_in + n_out + m) + (64 << 20)
    check(x.expand(m, T, n_in), w, a, b, sign[:, 0], 1)


@pytest.mark.parametrize('m,T,n_in,n_out', [(3, 70, 32, 8), (2, 33, 300, 19)])
def test_the_bf16_c_entry(m, T, n_in, n_out):
    """noise_lowrank_rows is the drop-in's narrow form on bf16 tensors, at any number of outputs: held to the same bound."""
    import ctypes
    from noise_amd import _lib
    x, w, a, b, sign = inputs(m, T, n_in, n_out, 2, torch.bfloat16, 7)
    wb, y = w.bfloat16(), torch.empty(m, T, n_out, device=DEV)
    pop = _lib.Population(m, T, sign.data_ptr(), 2)
    r1 = _lib.Rank1(a.data_ptr(), b.data_ptr(), n_out, n_in)
    _lib.call('noise_lowrank_rows', ctypes.byref(pop), _lib.View(x.data_ptr(), T * n_in, n_in), n_in, wb.data_ptr(), n_out,
              ctypes.byref(r1), y.data_ptr(), _lib.stream_ptr(DEV))
    check(x, wb, a, b, sign, 2, y)


@pytest.mark.parametrize('form', [0, 1, 2])
@pytest.mark.parametrize('K,N', [(512, 256), (192, 512)])
def test_the_tiled_c_entry(form, K, N):
    """noise_pop_linear with its rank-1 term, as bf16 (0), fp32 (1) and autocast's fp32 (2). The fp32 sum of the terms rounds
    by 2^-20 of their sizes; form 0 rounds the result once more, and form 2 the product and the dot (one bf16 ulp each)."""
    import ctypes
    from noise_amd import _lib
    m, T = 3, 512
    x, w, a, b, sign = inputs(m, T, K, N, 2, torch.bfloat16, 9)
    wb, bb = w.bfloat16(), b.bfloat16().float()
    d = torch.arange(m, device=DEV) // 2
    dots = (x.float() * bb[d][:, None, :]).sum(-1)
    y = torch.empty(m, T, N, device=DEV, dtype=torch.bfloat16 if form == 0 else torch.float32)
    pop = _lib.Population(m, T, sign.data_ptr(), 2)
    r1 = _lib.Rank1(a.data_ptr(), bb.data_ptr(), N, K)
    _lib.call('noise_pop_linear', ctypes.byref(pop), _lib.View(x.data_ptr(), T * K, K), wb.data_ptr(), K, N, ctypes.byref(r1),
              dots.data_ptr(), y.data_ptr(), form, T * N, N, _lib.stream_ptr(DEV))
    if form == 2:
        check(x, wb, a, b, sign, 2, y)
        return
    xd, wd = x.double(), wb.double()
    term = (sign[:, None] * dots).double()[..., None] * a.double()[d][:, None, :]
    ref = torch.stack([xd[i] @ wd.t() for i in range(m)]) + term
    size = torch.stack([xd[i].abs() @ wd.abs().t() for i in range(m)]) + term.abs()
    bound = size * 2.0 ** -20 + (ref.abs() * 2.0 ** -7 if form == 0 else 0)
    assert ((y.double() - ref).abs() <= bound).all()
