"""Steps of gated linear attention, HGRN2 and RWKV by workgroups of 512 and of
256 threads: states around the line between them, columns that do not divide
the threads."""

import pytest
import torch

import resilient_llm_amd.ops as ops
from nesizen_util import BF16, F32
from resilient_llm_amd.engine.batch import Portion, PromptRows
from test_lat_ops import hgrn2_case
from test_mix_ops import gla_case, rel, tol
from test_rec_ops import Rwkv


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("dim,vdim,rank", [
    (128, 256, 8), (127, 256, 24), (164, 200, 40), (256, 256, 64),
    (252, 130, 33)])
def test_steps(dim, vdim, rank, dtype):
    T, H = 9, 2
    *inputs, eps, want, S = gla_case(T, H, dim, vdim, rank, 8.0, 1.0,
                                     dim + rank, dtype)
    proj, a2, b, norm = (t.cuda() for t in inputs)
    st = torch.full((3, H, dim, -(-vdim // 4) * 4), float("nan"),
                    device="cuda")
    slot = torch.tensor([1], dtype=torch.int32, device="cuda")
    got = torch.cat([
        ops.gla_decode(proj[p:p + 1].contiguous(), a2, b, norm, st, slot,
                       torch.tensor([p], dtype=torch.int32, device="cuda"),
                       vdim, 8.0, eps) for p in range(T)])
    # the bounds of the longer runs over the same steps
    assert rel(got, want) < tol(dtype)
    assert rel(st[1, :, :, :vdim], S) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("dim,vdim", [(128, 256), (127, 256), (164, 200),
                                      (256, 256), (252, 130)])
def test_hgrn2_steps(dim, vdim, dtype):
    T, H = 9, 2
    *inputs, eps, want, S = hgrn2_case(T, H, dim, vdim, 1.0, 0.8, dim, dtype)
    proj, b, lower, norm = (t.cuda() for t in inputs)
    st = torch.full((3, H, dim, -(-vdim // 4) * 4), float("nan"),
                    device="cuda")
    slot = torch.tensor([1], dtype=torch.int32, device="cuda")
    got = torch.cat([
        ops.hgrn2_decode(proj[p:p + 1].contiguous(), b, lower, norm, st, slot,
                         torch.tensor([p], dtype=torch.int32, device="cuda"),
                         vdim, eps) for p in range(T)])
    assert rel(got, want) < tol(dtype)
    assert rel(st[1, :, :, :vdim], S) < 3e-5


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("dim", [180, 184, 255, 256])
def test_rwkv_steps(dim, dtype):
    T = 9
    a = Rwkv(T, 2, dim, 16, "cuda", dtype, seed=dim)
    want, S = a.want()
    got = torch.cat([a.call(p, 1, 1) for p in range(T)])
    # the bounds of the longer runs
    assert rel(got, want) < (1e-5 if dtype == F32 else 8e-3)
    assert rel(a.state[1, :, :, :a.dim].cpu(), S) < 2e-5


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("dim,vdim,rank", [
    # 512 threads from 128 x 128 on
    (128, 128, 16), (127, 128, 16), (256, 64, 4), (255, 64, 8),
    # 256 threads with four rows each, where that is all rows, or eight
    (64, 64, 16), (65, 64, 16), (16, 256, 68), (17, 256, 12), (1, 4, 4),
    # one to sixteen lanes a channel; ranks that fours do not divide and rows
    # that do not lie for them
    (8, 30, 64), (16, 33, 64), (33, 20, 20), (120, 40, 3), (7, 12, 70),
    (32, 7, 1), (200, 24, 130)])
def test_lanes_and_rows(dim, vdim, rank, dtype):
    T, H = 5, 3
    *inputs, eps, want, S = gla_case(T, H, dim, vdim, rank, 8.0, 1.0,
                                     dim + rank, dtype)
    proj, a2, b, norm = (t.cuda() for t in inputs)
    # rows of three sequences, whose other slots hold NaN
    st = torch.full((5, H, dim, -(-vdim // 4) * 4), float("nan"),
                    device="cuda")
    slots = torch.tensor([4, 0, 2], dtype=torch.int32, device="cuda")
    got = torch.stack([
        ops.gla_decode(proj[p:p + 1].repeat(3, 1), a2, b, norm, st, slots,
                       torch.full((3,), p, dtype=torch.int32, device="cuda"),
                       vdim, 8.0, eps) for p in range(T)])
    # the bounds of the longer runs over the same steps
    for i, slot in enumerate((4, 0, 2)):
        assert rel(got[:, i], want) < tol(dtype)
        assert rel(st[slot, :, :, :vdim], S) < 1e-5
    assert torch.isnan(st[[1, 3]]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("seqs,H,dim,vdim", [
    # slices of 16, 32 and 64 columns, full and ragged ones; odd numbers of
    # tiles down the columns
    (2, 3, 128, 48), (2, 3, 40, 33), (2, 64, 40, 33), (2, 64, 64, 32),
    (2, 64, 130, 40), (2, 64, 128, 128), (2, 64, 24, 97), (2, 64, 72, 70),
    # as many slices of 16, 32 and 64 columns as there are CUs, and one more head
    (2, 8, 128, 256), (2, 9, 64, 256), (2, 16, 128, 256), (2, 17, 128, 250),
    (2, 33, 64, 256), (1, 3, 256, 64), (2, 24, 256, 96), (2, 5, 144, 64),
    # some 60 MB of operands and all slices at once; more slices than CUs
    (2, 104, 128, 64), (4, 86, 96, 48), (4, 72, 128, 80),
    # short heads that fill the chip: f32 operands
    (4, 128, 16, 20), (4, 128, 64, 64)])
def test_prompts_by_slices(seqs, H, dim, vdim):
    lens = [130, 65, 3, 64][:seqs]
    *inputs, eps, want, S = gla_case(lens[0], H, dim, vdim, 8, 8.0, 1.0,
                                     dim + vdim, BF16)
    proj, a2, b, norm = (t.cuda() for t in inputs)
    st = torch.full((seqs + 1, H, dim, -(-vdim // 4) * 4), float("nan"),
                    device="cuda")
    portions, at = [], 0
    for i, n in enumerate(lens):
        portions.append(Portion(at, 0, n, i, i))
        at += n
    got = ops.gla_prefill(torch.cat([proj[:n] for n in lens]), a2, b, norm,
                          st, PromptRows(portions, "cuda"), vdim, 8.0, eps)
    # the bounds of the longer runs over the same steps
    for n, rows in zip(lens, got.split(lens)):
        assert rel(rows, want[:n]) < tol(BF16)
    assert rel(st[0, :, :, :vdim], S) < 1e-5
    assert torch.isnan(st[seqs]).all()


def scan_of(lens, H, dim, vdim):
    """Parts or f32, columns of a slice, and whether slices ask for lines ahead."""
    ops.load_libraries(("rlli_rec",))
    return torch.ops.rlli_rec.gla_scan(
        sum(lens), sum(-(-n // 64) for n in lens), len(lens), H, dim, vdim)


@pytest.mark.gpu
@pytest.mark.parametrize("seqs,H,dim,vdim,T,cols", [
    (8, 4, 128, 128, 1216, 16), (8, 4, 64, 128, 2400, 16),
    (8, 4, 128, 256, 1216, 32), (8, 4, 64, 256, 2400, 32),
    (11, 4, 128, 160, 900, 32), (11, 4, 64, 160, 1900, 32),
    (16, 4, 128, 256, 600, 64), (16, 4, 64, 192, 1100, 64),
    # one slice of a head
    (20, 8, 128, 64, 280, 64), (24, 8, 64, 64, 460, 64)])
def test_prompts_of_many_operands(seqs, H, dim, vdim, T, cols):
    """Some 60 MB of a scan's operands, lines of which slices ask for ahead of
    time: chunk counts that are even, odd and one."""
    lens = [T] * seqs
    lens[1], lens[2], lens[3] = T - 70, T - 1, 1
    assert scan_of(lens, H, dim, vdim) == [1, cols, 1]
    *inputs, eps, want, S = gla_case(T, H, dim, vdim, 8, 8.0, 1.0, dim, BF16)
    proj, a2, b, norm = (t.cuda() for t in inputs)
    st = torch.full((len(lens), H, dim, vdim), float("nan"), device="cuda")
    portions, at = [], 0
    for i, n in enumerate(lens):
        portions.append(Portion(at, 0, n, i, i))
        at += n
    got = ops.gla_prefill(torch.cat([proj[:n] for n in lens]), a2, b, norm,
                          st, PromptRows(portions, "cuda"), vdim, 8.0, eps)
    for i, (n, rows) in enumerate(zip(lens, got.split(lens))):
        assert rel(rows, want[:n]) < tol(BF16)
        if n == T:
            assert rel(st[i], S) < 1e-5


@pytest.mark.parametrize("seqs,H,dim,vdim,T,form", [
    # heads of more than 128: f32 operands where many fill the chip
    (4, 64, 132, 72, 70, 0), (2, 64, 132, 256, 66, 1), (1, 32, 132, 33, 3100, 1),
    # up to 64 columns: where they fill it and are 48 Ki rows of all heads, or 96 Ki
    # on up to 128 workgroups
    (8, 64, 128, 40, 97, 0), (8, 64, 100, 33, 95, 1), (2, 16, 72, 20, 3100, 0),
    (2, 16, 72, 20, 3000, 1), (9, 16, 128, 64, 700, 1),
    # more columns: where they fill it and up to 128
    (2, 16, 72, 100, 3100, 1), (8, 64, 100, 128, 97, 0), (8, 64, 100, 130, 97, 1),
    # short heads that fill it
    (8, 64, 64, 64, 10, 0), (7, 64, 64, 64, 10, 1)])
def test_form_of_the_scans_operands(seqs, H, dim, vdim, T, form):
    assert scan_of([T] * seqs, H, dim, vdim)[0] == form


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, BF16])
def test_infinite_state(dtype):
    """One infinite number of a state makes its column infinite, whatever its
    sign and the queries, and the norm the head's other columns zero; no other
    head sees it."""
    T, H, dim, vdim, at = 70, 3, 64, 96, 37
    *inputs, eps, want, S = gla_case(T, H, dim, vdim, 8, 8.0, 1.0, 5, dtype)
    proj, a2, b, norm = (t.cuda() for t in inputs)
    st = torch.zeros(1, H, dim, vdim, device="cuda")
    clean = st.clone()
    st[0, 1, 9, at] = float("-inf")
    rows = PromptRows([Portion(0, 64, T, 0, 0)], "cuda")
    got, ref = (ops.gla_prefill(proj, a2, b, norm, s, rows, vdim, 8.0,
                                eps).view(T, H, vdim) for s in (st, clean))
    assert torch.equal(got[:, 0], ref[:, 0])
    assert torch.equal(got[:, 2], ref[:, 2])
    rest = torch.arange(vdim, device="cuda") != at
    assert not torch.isfinite(got[:, 1, at]).any()
    assert (got[:, 1][:, rest] == 0).all()
    assert torch.isinf(st[0, 1, 9, at])
    st[0, 1, 9, at] = clean[0, 1, 9, at]
    assert torch.equal(st, clean)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("row", [1, 9, 17, 40, 63])
def test_nothing_of_later_rows(row, dtype):
    """Values as large as there are leave the bits of small rows ahead of them as
    they are."""
    T, H, dim, vdim = 64, 2, 64, 32
    proj, a2, b, norm = (t.cuda() for t in gla_case(T, H, dim, vdim, 8, 8.0, 1.0,
                                                    5, dtype)[:4])
    proj[:row] *= 2.0 ** -20
    loud = proj.clone()
    loud[row:, 2 * H * dim:2 * H * dim + H * vdim] = 2.0 ** 126
    got, want = (ops.gla_prefill(
        p, a2, b, norm, torch.zeros(1, H, dim, vdim, device="cuda"),
        PromptRows([Portion(0, 0, T, 0, 0)], "cuda"), vdim, 8.0, 1e-30)[:row]
        for p in (loud, proj))
    assert want.isfinite().all() and (want != 0).any()
    assert torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 15, 63, 64, 65, 130])
@pytest.mark.parametrize("dim,rank", [(64, 16), (128, 16), (128, 48), (64, 24)])
def test_prompts_without_conditions(T, dim, rank):
    """Heads of 64 and 128 whose rows and ranks come in whole loads, up to and
    beyond a chunk's last row."""
    H, vdim = 2, 48
    *inputs, eps, want, S = gla_case(T, H, dim, vdim, rank, 8.0, 1.0, T + rank,
                                     BF16)
    # what lies behind the last row is not a row
    proj, a2, b, norm = (t.cuda() for t in inputs)
    proj = torch.cat([proj, torch.full_like(proj[:1], float("nan"))])[:T]
    st = torch.full((2, H, dim, vdim), float("nan"), device="cuda")
    got = ops.gla_prefill(proj, a2, b, norm, st,
                          PromptRows([Portion(0, 0, T, 0, 1)], "cuda"), vdim,
                          8.0, eps)
    # the bounds of the longer runs over the same steps
    assert rel(got, want) < tol(BF16)
    assert rel(st[1], S) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,seqs,dim,each", [
    (BF16, 16, 64, 4), (BF16, 15, 64, 6), (BF16, 2, 128, 6), (F32, 2, 128, 4),
    (BF16, 32, 128, 4), (BF16, 16, 256, 4), (BF16, 8, 256, 6)])
def test_scratch_of_prompts(dtype, seqs, dim, each):
    """As many bytes as the scan's operands have: four a number where they are f32,
    as of heads that fill the chip, or three parts."""
    H, vdim, T = 32, 64, 64
    rows = PromptRows([Portion(i * T, 0, T, i, i) for i in range(seqs)], "cuda")
    proj = torch.zeros(T * seqs, 2 * H * (dim + vdim) + 8, device="cuda",
                       dtype=dtype)
    a2 = torch.zeros(H * dim, 8, device="cuda", dtype=dtype)
    st = torch.zeros(seqs, H, dim, vdim, device="cuda")
    args = (proj, a2, torch.zeros(H * dim, device="cuda"),
            torch.ones(vdim, device="cuda"), st, rows, vdim, 8.0, 1e-5)
    ops.gla_prefill(*args)                # (makes the tables)
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    out = ops.gla_prefill(*args)
    took = torch.cuda.max_memory_allocated() - before
    chunks = H * seqs
    want = (chunks * (64 * dim * 2 + 64 * 64) * each + chunks * dim * 4
            + (T * seqs + 64) * H * vdim * 4 + out.nbytes)
    # (each of six allocations may have a block that is up to 1 MB larger; with six
    # bytes for four the first case would take 12 MB more)
    assert took <= want + (6 << 20)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["gla", "hgrn2", "rwkv"])
@pytest.mark.parametrize("seqs,H,dim,vdim,T", [
    # heads of more than 128: f32 operands where many fill the chip
    (4, 64, 132, 72, 70), (2, 64, 132, 256, 66),
    # of up to 128: from 48 Ki rows of all heads on where they fill it; 96 Ki
    # elsewhere, but not of more than 64 columns, nor wide ones
    (8, 64, 128, 40, 97), (8, 64, 100, 33, 95), (2, 16, 72, 20, 3100),
    (1, 32, 132, 33, 3100), (2, 16, 72, 100, 3100), (8, 64, 100, 128, 97),
    (8, 64, 100, 130, 97)])
def test_prompts_of_many_heads(seqs, H, dim, vdim, T, kind):
    """Both sides of the lines where the scan's operands are f32 and not parts."""
    rows = PromptRows([Portion(i * T, 0, T, i, i) for i in range(seqs)], "cuda")
    cuda = lambda *ts: [t.cuda() for t in ts]
    if kind == "rwkv":
        vdim = dim
        a = Rwkv(T, H, dim, 8, "cpu", BF16, seed=dim)
        want, S = a.want()
    elif kind == "gla":
        *inputs, eps, want, S = gla_case(T, H, dim, vdim, 8, 8.0, 1.0,
                                         dim + vdim, BF16)
    else:
        *inputs, eps, want, S = hgrn2_case(T, H, dim, vdim, 1.0, 0.8, dim, BF16)
    st = torch.full((seqs + 1, H, dim, -(-vdim // 4) * 4), float("nan"),
                    device="cuda")
    if kind == "rwkv":
        got = torch.full((seqs * T, H * dim), float("nan"), device="cuda",
                         dtype=BF16)
        ops.rwkv_prefill(
            a.rkvg.repeat(1, seqs, 1).cuda(), a.low.repeat(seqs, 1).cuda(),
            *cuda(a.w2, a.w0, a.u, a.norm), st, rows, a.eps, got)
    else:
        proj, *rest = cuda(*inputs)
        proj = proj.repeat(seqs, 1)
        got = ops.gla_prefill(proj, *rest, st, rows, vdim, 8.0, eps) \
            if kind == "gla" else \
            ops.hgrn2_prefill(proj, *rest, st, rows, vdim, eps)
    # the bounds of the longer runs over the same steps
    for i, of in enumerate(got.split(T)):
        assert rel(of, want) < (8e-3 if kind == "rwkv" else tol(BF16))
        assert rel(st[i, :, :, :vdim], S) < \
            {"gla": 1e-5, "hgrn2": 3e-5, "rwkv": 2e-5}[kind]
    assert torch.isnan(st[seqs]).all()
