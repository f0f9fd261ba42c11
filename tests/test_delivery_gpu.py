"""The GEMM's epilogue as the groups' consumer: a call in the automatic mode, which delivers every group up to
K = 8192 and above it those that complete with the GEMM, against the same call with every group waited for and
copied (consumer mode 1).  The same tiles take another way to the same place, so every buffer has to be
bit-identical, and the counters have to end at zero either way.  released_groups() says which way they took."""
import ctypes as C

import pytest
import torch

import flashoverlap_amd
from flashoverlap_amd import capi, tiling

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def api(dev):
    flashoverlap_amd.load()
    capi.check(capi.lib().fo_set_wait_timeout_ms(5000))
    return torch.classes.flashoverlap_class


def _object(api, mode, rank=0, size=1):
    o = api.OverlapImpl()
    o.mccl_init(rank, size, torch.ops.flashoverlap_op.generate_mccl_id())
    o.mutlass_init()
    o.overlap_init()
    o.set_consumer_mode(mode)
    return o


def _inputs(dev, dt, M, N, K):
    g = torch.Generator(device=dev).manual_seed(M + 3 * N + 7 * K)
    return tuple((torch.randn(r, K, generator=g, device=dev) / K ** 0.25).to(dt) for r in (M, N))


def _released(mode, M, N, K, algo, cseg):
    """The groups of a call that go through their counters: in the automatic mode none up to K = 8192, and above
    it those with a tile in front of the last round of workgroups, but for the last one."""
    if mode:
        return len(cseg)
    if K <= 8192:
        return 0
    per, late = C.c_int(), C.c_int()
    capi.check(capi.lib().fo_gemm_rounds(algo, M, N, C.byref(per), C.byref(late)))
    return sum(sum(cseg[:g]) < late.value for g in range(len(cseg) - 1))


@pytest.mark.parametrize("M,N,K,algo,cseg", [
    (128, 128, 64, 1, [1]),                      # one tile
    (384, 640, 328, 1, [4, 0, 11]),              # odd multiples of 128, an empty group, a partial last panel
    (512, 768, 128, 2, [5, 7]),                  # 128x256 layout tiles: half macro tiles and whole ones
    (768, 384, 72, 4, [1] * 9),                  # 256x128
    (8192, 2304, 64, 1, [600, 424, 64, 64]),     # 288 macro tiles of 256: a first round and 32 tiles of a second
    (8192, 2304, 8200, 1, [600, 424, 64, 64]),   # the same with the groups of the first round released
])
@pytest.mark.parametrize("ws,stacked", [(1, False), (4, False), (8, True)])
def test_delivered_groups_equal_copied_groups(api, dev, M, N, K, algo, cseg, ws, stacked):
    print(f"delivery {M}x{N}x{K} algo {algo} ws {ws} stacked {stacked}", flush=True)
    dt = torch.bfloat16
    BM, BN, _ = capi.algo_tile(algo)
    TM, TN = M // BM, N // BN
    cs = torch.tensor(cseg, dtype=torch.int32)
    RA = tiling.reorder_indices(TM * TN, tiling.raster_hint(M, N, algo), dev).reshape(TM, TN)
    RE = tiling.generate_row_remap_array(M, N, BM, BN, cseg, ws, dev) if ws > 1 else None
    A, B = _inputs(dev, dt, M, N, K)
    got = []
    for mode in (1, 0):
        o = _object(api, mode, ws - 1, ws)
        mm = torch.zeros(len(cseg), dtype=torch.int32, device=dev)
        c = torch.full((M, N), 7.0, dtype=dt, device=dev)
        d = torch.full(((ws if stacked else 1) * M // ws, N), 7.0, dtype=dt, device=dev)
        torch.cuda.synchronize()
        for _ in range(2):     # the second call finds the first one's counters
            if ws > 1:
                o.gemm_reducescatter_overlap(A, B, c, d, mm, RA, RE, 1, cs, cs.to(dev), algo, False)
            else:
                o.set_staging(d)
                o.gemm_allreduce_overlap(A, B, c, mm, RA, 1, cs, cs.to(dev), algo, False)
        torch.cuda.synchronize()
        assert o.wait_timeouts(True) == 0 and not mm.any()
        assert o.released_groups() == _released(mode, M, N, K, algo, cseg)
        got.append((c, d))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (127, 129, 72), (300, 520, 136), (384, 640, 64), (2049, 2056, 64)])
def test_serial_call_delivers_what_it_stores(api, dev, M, N, K):
    """gemm_allreduce: C and the staging buffer are both the plain GEMM's result, and nothing around them is touched."""
    A, B = _inputs(dev, torch.float16, M, N, K)
    want = torch.empty(M, N, dtype=torch.float16, device=dev)
    c = torch.empty_like(want)
    guard = torch.full((64 + M * N + 64,), 7.0, dtype=torch.float16, device=dev)
    staging = guard[64:64 + M * N]
    o = _object(api, 0)
    o.mutlass_gemm(A, B, want, 1)
    o.set_staging(staging)
    o.gemm_allreduce(A, B, c, 1)
    torch.cuda.synchronize()
    assert torch.equal(c, want) and torch.equal(staging.view(M, N), want)
    assert (guard[:64] == 7.0).all() and (guard[64 + M * N:] == 7.0).all()
    # a staging buffer that is also an operand is written only when the GEMM has read it
    if M * N <= A.numel():
        o.set_staging(A.view(-1)[:M * N])
        o.gemm_allreduce(A, B, c, 1)
        torch.cuda.synchronize()
        assert torch.equal(c, want) and torch.equal(A.view(-1)[:M * N].view(M, N), want)


def test_rounds_of_a_shape(dev):
    """288 macro tiles on 256 CUs: the last round starts at macro tile 256, layout tile 1024 in issue order."""
    per, late, cus = C.c_int(), C.c_int(), C.c_int()
    rounds = capi.lib().fo_gemm_rounds
    capi.check(capi.lib().fo_device_info(C.byref(cus), None, None))
    capi.check(rounds(1, 8192, 2304, C.byref(per), C.byref(late)))
    if cus.value == 256:
        assert (per.value, late.value) == (1024, 1024)
    capi.check(rounds(1, 1024, 1024, C.byref(per), C.byref(late)))
    assert late.value == 0
    assert rounds(1, 100, 1024, C.byref(per), C.byref(late)) == capi.FO_ERR_SHAPE


@pytest.mark.parametrize("ws,stacked", [(1, False), (4, False), (4, True)])
@pytest.mark.parametrize("group", [13, 100, 700])
def test_groups_of_a_round_released_together(api, dev, ws, stacked, group):
    """Two whole rounds and a bit, and a K above that with which every group is delivered: the groups of a round take
    one wait and one copy launch; with 13 tiles to a group there are more groups to a round than lanes to a wavefront."""
    M, N, K, algo, dt = 8192, 4352, 8200, 1, torch.float16
    BM, BN, _ = capi.algo_tile(algo)
    TM, TN = M // BM, N // BN
    cseg = tiling.uniform_cseg(TM * TN, group)
    cs = torch.tensor(cseg, dtype=torch.int32)
    RA = tiling.reorder_indices(TM * TN, tiling.raster_hint(M, N, algo), dev).reshape(TM, TN)
    RE = tiling.generate_row_remap_array(M, N, BM, BN, cseg, ws, dev) if ws > 1 else None
    A, B = _inputs(dev, dt, M, N, K)
    got = []
    for mode in (1, 0):
        o = _object(api, mode, ws - 2 if ws > 1 else 0, ws)
        mm = torch.zeros(len(cseg), dtype=torch.int32, device=dev)
        c = torch.full((M, N), 7.0, dtype=dt, device=dev)
        d = torch.full(((ws if stacked else 1) * M // ws, N), 7.0, dtype=dt, device=dev)
        o.set_staging(d)
        torch.cuda.synchronize()
        for _ in range(2):
            if ws > 1:
                o.gemm_reducescatter_overlap(A, B, c, d, mm, RA, RE, 1, cs, cs.to(dev), algo, False)
            else:
                o.gemm_allreduce_overlap(A, B, c, mm, RA, 1, cs, cs.to(dev), algo, False)
        torch.cuda.synchronize()
        assert o.wait_timeouts(True) == 0 and not mm.any()
        assert o.released_groups() == _released(mode, M, N, K, algo, cseg)
        got.append((c, d))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("M,N,K,cseg", [
    (1024, 1024, 512, [16, 16, 0, 20, 12]),      # one round: all of it would be delivered
    (8192, 2304, 64, [300, 300, 424, 64, 64]),   # groups of a round, and a last round
])
@pytest.mark.parametrize("ws,rank", [(2, 1), (4, 0), (4, 3)])
def test_receive_buffer_in_the_first_rows_of_c(api, dev, M, N, K, cseg, ws, rank):
    """D = C[:M / ws]: a group's rows are written over rows of groups that are complete, one group after the other."""
    algo, dt = 1, torch.bfloat16
    print(f"D in C {M}x{N}x{K} rank {rank} of {ws}", flush=True)
    BM, BN, _ = capi.algo_tile(algo)
    TM, TN = M // BM, N // BN
    cs = torch.tensor(cseg, dtype=torch.int32)
    RA = tiling.reorder_indices(TM * TN, tiling.raster_hint(M, N, algo), dev).reshape(TM, TN)
    RE = tiling.generate_row_remap_array(M, N, BM, BN, cseg, ws, dev)
    A, B = _inputs(dev, dt, M, N, K)
    o = _object(api, 0, rank, ws)
    mm = torch.zeros(len(cseg), dtype=torch.int32, device=dev)
    want_c, want_d = torch.empty(M, N, dtype=dt, device=dev), torch.empty(M // ws, N, dtype=dt, device=dev)
    o.gemm_reducescatter_overlap(A, B, want_c, want_d, mm, RA, RE, 1, cs, cs.to(dev), algo, False)
    for mode in (0, 1):
        o.set_consumer_mode(mode)
        for _ in range(3):
            c = torch.full((M, N), 7.0, dtype=dt, device=dev)
            o.gemm_reducescatter_overlap(A, B, c, c[:M // ws], mm, RA, RE, 1, cs, cs.to(dev), algo, False)
            torch.cuda.synchronize()
            assert o.wait_timeouts(True) == 0 and not mm.any()
            assert torch.equal(c[:M // ws], want_d) and torch.equal(c[M // ws:], want_c[M // ws:])


@pytest.mark.parametrize("M,N,K,group", [(1024, 1024, 512, 8), (8192, 2304, 64, 200), (128, 4096, 4096, 8),
                                         (8192, 2304, 8200, 200)])   # the last: groups of the first round released
def test_all_reduce_in_place(api, dev, M, N, K, group):
    """The staging buffer is C itself, with and without overlap: C is what it is with a buffer of its own."""
    algo, dt = 1, torch.float16
    BM, BN, _ = capi.algo_tile(algo)
    TM, TN = M // BM, N // BN
    cseg = tiling.uniform_cseg(TM * TN, group)
    cs = torch.tensor(cseg, dtype=torch.int32)
    RA = tiling.reorder_indices(TM * TN, tiling.raster_hint(M, N, algo), dev).reshape(TM, TN)
    A, B = _inputs(dev, dt, M, N, K)
    o = _object(api, 0)
    mm = torch.zeros(len(cseg), dtype=torch.int32, device=dev)
    got = []
    for in_place in (False, True):
        c = torch.full((2, M, N), 7.0, dtype=dt, device=dev)
        other = torch.empty(M, N, dtype=dt, device=dev)
        o.set_staging(c[0] if in_place else other)
        o.gemm_allreduce_overlap(A, B, c[0], mm, RA, 1, cs, cs.to(dev), algo, False)
        torch.cuda.synchronize()
        o.set_staging(c[1] if in_place else other)
        o.gemm_allreduce(A, B, c[1], algo)
        torch.cuda.synchronize()
        assert o.wait_timeouts(True) == 0 and not mm.any()
        assert o.released_groups() == _released(0, M, N, K, algo, cseg)
        got.append(c)
    assert torch.equal(got[0], got[1])


@pytest.mark.parametrize("M,N,K,group", [
    (8192, 4352, 8192, 100),     # the longest K with which every group is delivered
    (8192, 4352, 8200, 100),     # and one above it: the groups of the first rounds are waited for, round by round
    (16384, 8192, 72, 1000),     # delivered, 256 MiB of output: stored past the caches
])
@pytest.mark.parametrize("ws", [1, 4])
def test_which_groups_are_delivered(api, dev, M, N, K, group, ws):
    algo, dt = 1, torch.bfloat16
    print(f"delivery rule {M}x{N}x{K} ws {ws}", flush=True)
    BM, BN, _ = capi.algo_tile(algo)
    TM, TN = M // BM, N // BN
    cseg = tiling.uniform_cseg(TM * TN, group)
    cs = torch.tensor(cseg, dtype=torch.int32)
    RA = tiling.reorder_indices(TM * TN, tiling.raster_hint(M, N, algo), dev).reshape(TM, TN)
    RE = tiling.generate_row_remap_array(M, N, BM, BN, cseg, ws, dev) if ws > 1 else None
    A, B = (torch.empty(r, K, dtype=dt, device=dev).normal_() for r in (M, N))
    got = []
    for mode in (1, 0):
        o = _object(api, mode, ws - 1, ws)
        mm = torch.zeros(len(cseg), dtype=torch.int32, device=dev)
        c = torch.full((M, N), 7.0, dtype=dt, device=dev)
        d = torch.full((M // ws, N), 7.0, dtype=dt, device=dev)
        o.set_staging(d)
        torch.cuda.synchronize()
        if ws > 1:
            o.gemm_reducescatter_overlap(A, B, c, d, mm, RA, RE, 1, cs, cs.to(dev), algo, False)
        else:
            o.gemm_allreduce_overlap(A, B, c, mm, RA, 1, cs, cs.to(dev), algo, False)
        torch.cuda.synchronize()
        assert o.wait_timeouts(True) == 0 and not mm.any()
        assert o.released_groups() == _released(mode, M, N, K, algo, cseg)
        got.append((c, d))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("M,N,K,algo", [(128, 128, 64, 1), (384, 640, 328, 1), (512, 768, 128, 2), (768, 384, 72, 4),
                                        (128, 1024, 4096, 1), (4352, 4096, 520, 1)])
@pytest.mark.parametrize("ws,kept", [(1, 1), (4, 1), (4, 4)])
def test_delivered_without_c(dev, M, N, K, algo, ws, kept):
    """fo_gemm_deliver stores what fo_gemm_launch delivers, and nothing else; with and without a split over K."""
    L, dt = capi.lib(), torch.float16
    BM, BN, _ = capi.algo_tile(algo)
    T = (M // BM) * (N // BN)
    cseg = tiling.uniform_cseg(T, max(1, T // 3))
    start = [sum(cseg[:g]) for g in range(len(cseg))]
    cs, st = (torch.tensor(v, dtype=torch.int32, device=dev) for v in (cseg, start))
    table = torch.repeat_interleave(torch.arange(len(cseg), dtype=torch.int32, device=dev), cs.long()).int()
    RA = tiling.reorder_indices(T, tiling.raster_hint(M, N, algo), dev)
    RE = tiling.generate_row_remap_array(M, N, BM, BN, cseg, ws, dev)
    mm = torch.zeros(len(cseg), dtype=torch.int32, device=dev)
    A, B = _inputs(dev, dt, M, N, K)
    D = torch.full((M * N,), 7.0, dtype=dt, device=dev)
    got = []
    for entry in (L.fo_gemm_launch, L.fo_gemm_deliver):
        out = torch.full((M * N * kept // ws + 64,), 7.0, dtype=dt, device=dev)
        c = capi.GemmCall(mode=2 if ws > 1 else 1, dtype=capi.FO_F16, algo=algo, M=M, N=N, K=K, rLDN=1, cseg_dev=cs.data_ptr(),
                          G=len(cseg), group_table=table.data_ptr(), A=A.data_ptr(), B=B.data_ptr(), MM=mm.data_ptr(),
                          RA=RA.data_ptr(), RE=RE.data_ptr(), deliver=out.data_ptr(), nslices=ws, slice_first=0 if kept == ws else 2,
                          slice_count=kept, slice_stride=M * N // ws, group_start=st.data_ptr())
        if entry is L.fo_gemm_launch:
            c.D = D.data_ptr()
        need = C.c_size_t()
        capi.check(L.fo_gemm_workspace(C.byref(c), C.byref(need)))
        work = torch.zeros(need.value // 4 + 1, device=dev)
        c.workspace, c.workspace_bytes = work.data_ptr(), need.value
        capi.check(entry(C.byref(c), None))
        torch.cuda.synchronize()
        assert not mm.any() and (out[-64:] == 7.0).all()
        got.append(out)
    assert torch.equal(got[0], got[1])
    c.deliver_from = 1                      # a tile that is not delivered would be lost
    assert L.fo_gemm_deliver(C.byref(c), None) == capi.FO_ERR_ARG
    c.deliver_from, c.mode = 0, 0
    assert L.fo_gemm_deliver(C.byref(c), None) == capi.FO_ERR_ARG
    assert L.fo_gemm_deliver(None, None) == capi.FO_ERR_ARG
