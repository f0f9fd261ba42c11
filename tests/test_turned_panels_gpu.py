"""256x128 tiles whose XCDs begin at eight places of K (turn_panels, fo_plan.h), and tiles on the other side of each edge of that rule, in
every mode of the kernel.  Small whole numbers as operands make every fp32 sum exact, so that the result is its rounding whatever the
order; operands that are not whole are held against sums in 64 bits."""
import ctypes as C
import os
import subprocess

import pytest
import torch

import flashoverlap_amd
from flashoverlap_amd import capi, tiling

HERE = os.path.dirname(os.path.abspath(__file__))

# (M, N, K): panels between two places
PLAIN = {
    (2048, 2048, 3072): 6, (2048, 2048, 3136): 6, (2048, 2048, 3520): 6, (2048, 2048, 4096): 8,   # 48 panels, 49, 55, 64
    (2048, 4096, 3520): 6, (512, 3968, 8128): 15,                          # a full round of 256 tiles, 127 panels
    (1152, 2176, 3520): 6, (1800, 1600, 3520): 6, (456, 4095, 3136): 6,    # a half tile, ragged tiles, unaligned rows of D
    (2048, 2048, 3008): 0, (2048, 2048, 3080): 0, (4224, 2048, 3520): 0,   # 47 panels, a partial last one, more tiles than a round has
    (2304, 2048, 3520): 0, (1800, 1544, 3520): 0,                          # a band on one XCD, a thin last column of tiles
}
# (M, N, K, Algo)
PLACED = {(2048, 2048, 3072, 1): 6, (2048, 2048, 3520, 4): 6, (1152, 2176, 3136, 1): 6, (2560, 2304, 8128, 1): 15, (2304, 2048, 3520, 1): 0}


def test_the_shapes_lie_where_they_say(tmp_path):
    exe = str(tmp_path / "turn_choice")
    csrc = os.path.join(HERE, "..", "flashoverlap_amd", "csrc")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", csrc, os.path.join(HERE, "turn_choice.cpp"), "-o", exe], check=True)
    asked = {**PLAIN, **{s[:3]: panels for s, panels in PLACED.items()}}
    said = subprocess.run([exe], input="".join("%d %d %d\n" % s for s in asked), capture_output=True, text=True, check=True).stdout
    assert [int(line.split()[0]) for line in said.splitlines()] == list(asked.values())


@pytest.fixture
def tall():
    capi.check(capi.lib().fo_tune(b"macro_tile", 256128))
    yield
    capi.check(capi.lib().fo_tune(b"macro_tile", 0))


def _object():
    flashoverlap_amd.load()
    o = torch.classes.flashoverlap_class.OverlapImpl()
    o.mccl_init(0, 1, torch.ops.flashoverlap_op.generate_mccl_id())
    o.mutlass_init()
    o.overlap_init()
    return o


def _operands(m, n, k, dtype, dev):
    g = torch.Generator(device=dev).manual_seed(m + n + k)
    a, b = (torch.randint(-3, 4, (r, k), generator=g, device=dev).to(dtype) for r in (m, n))
    return a, b, (a.float() @ b.float().t()).to(dtype)


def _by_slot(want, ra, bm, bn):
    """The tiles of a row-major matrix, in the order of their slots."""
    tm, tn = want.size(0) // bm, want.size(1) // bn
    tiles = torch.empty(tm * tn, bm, bn, dtype=want.dtype, device=want.device)
    tiles[ra.flatten().long()] = want.reshape(tm, bm, tn, bn).transpose(1, 2).reshape(tm * tn, bm, bn)
    return tiles


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", list(PLAIN))
def test_every_panel_is_multiplied_once(m, n, k, dtype, dev, tall):
    a, b, want = _operands(m, n, k, dtype, dev)
    c, staging = (torch.full((m, n), float("nan"), dtype=dtype, device=dev) for _ in range(2))
    o = _object()
    o.set_staging(staging)
    o.gemm_allreduce(a, b, c, 1)
    assert torch.equal(c, want) and torch.equal(staging, want)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("consumer", [0, 1])   # delivered by the epilogue; released and copied
@pytest.mark.parametrize("m,n,k,algo", list(PLACED))
def test_signalled_tiles(m, n, k, algo, consumer, dtype, dev, tall):
    o = _object()
    o.set_consumer_mode(consumer)
    a, b, want = _operands(m, n, k, dtype, dev)
    bm, bn, _ = capi.algo_tile(algo)
    tm, tn = m // bm, n // bn
    cseg = tiling.uniform_cseg(tm * tn, 50)
    ra = tiling.reorder_indices(tm * tn, tiling.raster_hint(m, n, algo), dev).reshape(tm, tn)
    cseg_cpu = torch.tensor(cseg, dtype=torch.int32)
    counters = torch.zeros(len(cseg), dtype=torch.int32, device=dev)
    c, staging = (torch.full((m, n), float("nan"), dtype=dtype, device=dev) for _ in range(2))
    o.set_staging(staging)
    o.gemm_allreduce_overlap(a, b, c, counters, ra, 1, cseg_cpu, cseg_cpu.to(dev), algo, False)
    torch.cuda.synchronize()
    placed = _by_slot(want, ra, bm, bn)
    assert torch.equal(c.flatten(), placed.flatten()) and torch.equal(staging.flatten(), placed.flatten())
    assert int(counters.abs().sum()) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k,algo", list(PLACED))
def test_scattered_tiles(m, n, k, algo, dtype, dev, tall):
    """The first half of the groups signalled, the others delivered to four receive buffers."""
    world = 4
    a, b, want = _operands(m, n, k, dtype, dev)
    bm, bn, _ = capi.algo_tile(algo)
    t = (m // bm) * (n // bn)
    ra = tiling.reorder_indices(t, tiling.raster_hint(m, n, algo), dev)
    cseg = tiling.uniform_cseg(t, max(1, t // 6))
    start = [sum(cseg[:g]) for g in range(len(cseg))]
    half = len(cseg) // 2
    cs, st = (torch.tensor(v, dtype=torch.int32, device=dev) for v in (cseg, start))
    table = torch.repeat_interleave(torch.arange(len(cseg), device=dev), cs.long()).int()
    counters = torch.zeros(len(cseg), dtype=torch.int32, device=dev)
    re = tiling.generate_row_remap_array(m, n, bm, bn, cseg, world, dev)
    d, recv = (torch.full((t * bm, bn), 7.0, dtype=dtype, device=dev) for _ in range(2))
    unused = torch.zeros(4096, dtype=torch.uint8, device=dev)   # these tiles are not split; without one K is not begun apart
    call = capi.GemmCall(mode=2, dtype=capi.dtype_code(dtype), algo=algo, M=m, N=n, K=k, rLDN=1, A=a.data_ptr(), B=b.data_ptr(),
                         D=d.data_ptr(), cseg_dev=cs.data_ptr(), G=len(cseg), group_table=table.data_ptr(), MM=counters.data_ptr(),
                         RA=ra.data_ptr(), RE=re.data_ptr(), deliver=recv.data_ptr(), deliver_from=start[half], nslices=world,
                         slice_count=world, slice_stride=m * n // world, group_start=st.data_ptr(),
                         workspace=unused.data_ptr(), workspace_bytes=unused.nbytes)
    capi.check(capi.lib().fo_gemm_launch(C.byref(call), None))
    torch.cuda.synchronize()
    assert counters.cpu().tolist() == cseg[:half] + [0] * (len(cseg) - half)
    rows = torch.empty(t * bm, bn, dtype=dtype, device=dev)
    rows[re.long()] = _by_slot(want, ra, bm, bn).view(t * bm, bn)
    assert torch.equal(d, rows)
    expected = torch.full((world, t * bm // world, bn), 7.0, dtype=dtype, device=dev)
    for g in range(half, len(cseg)):
        first, count = start[g] * bm, cseg[g] * bm
        expected[:, first // world:(first + count) // world] = rows[first:first + count].view(world, count // world, bn)
    assert torch.equal(recv.view_as(expected), expected)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(1152, 2176, 3520), (456, 4095, 3136)])
def test_sums_in_another_order(m, n, k, dtype, dev, tall):
    """In whatever order K products are added in fp32, the sum is off by at most K 2^-24 of the sum of their absolute values; it is
    rounded once to the storage type.  A repeated call gives the same bits."""
    g = torch.Generator(device=dev).manual_seed(k)
    a = torch.randn(m, k, generator=g, device=dev).to(dtype)
    b = (0.02 * torch.randn(n, k, generator=g, device=dev)).to(dtype)
    out = [torch.full((m, n), float("nan"), dtype=dtype, device=dev) for _ in range(2)]
    o = _object()
    for c in out:
        o.mutlass_gemm(a, b, c, 1)
    assert torch.equal(*out)
    exact = a.cpu().double() @ b.cpu().double().t()
    summed = k * 2.0 ** -24 * (a.cpu().double().abs() @ b.cpu().double().abs().t())
    # (an fp16 result below 2^-14 is rounded to a multiple of 2^-24)
    rounded = (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8) * (exact.abs() + summed) + (2.0 ** -25 if dtype == torch.float16 else 0.0)
    assert ((out[0].cpu().double() - exact).abs() <= summed + rounded).all()
