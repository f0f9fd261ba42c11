"""Tiles split over K: the same GEMM with a workspace, through the C ABI, on integer-valued inputs (sums
are exact in fp32 whatever the order) against the product in fp32.  Shapes at the edges of the rule that
splits: one tile and many parts, edge tiles, a partial last panel in the last part, a last round of
256x256 tiles behind a whole one, half macro tiles."""
import ctypes as C

import pytest
import torch

from flashoverlap_amd import capi, tiling

pytestmark = pytest.mark.gpu

GUARD = 256


def _call(mode, dt, algo, A, B, D, **more):
    c = capi.GemmCall(mode=mode, dtype=capi.dtype_code(dt), algo=algo, M=A.size(0), N=B.size(0), K=A.size(1), rLDN=1,
                      A=A.data_ptr(), B=B.data_ptr(), D=D.data_ptr(), nslices=1)
    for k, v in more.items():
        setattr(c, k, v)
    need = C.c_size_t()
    capi.check(capi.lib().fo_gemm_workspace(C.byref(c), C.byref(need)))
    ws = torch.full((need.value // 4 + GUARD,), 1e30, dtype=torch.float32, device=D.device)
    ws[:1024] = 0
    c.workspace, c.workspace_bytes = ws.data_ptr(), need.value
    return c, ws, need.value


def _operands(dev, dt, M, N, K):
    g = torch.Generator().manual_seed(M + 3 * N + 7 * K)
    A, B = (torch.randint(-2, 3, (r, K), generator=g).to(dt).to(dev) for r in (M, N))
    return A, B, (A.float() @ B.float().t()).to(dt)


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [
    (128, 128, 8192),      # one tile
    (33, 129, 4104),       # four edge tiles, rows of D unaligned, 8 k in the last panel
    (100, 1160, 7168), (128, 4096, 4096), (256, 2048, 4160),
    (4352, 4096, 1544),    # 272 macro tiles of 256x256: sixteen behind a whole round
    (4225, 4104, 1984),    # 17 x 17: the tail is ragged in both directions
])
def test_split_plain(dev, dt, M, N, K):
    print(f"split {dt} {M}x{N}x{K}", flush=True)
    A, B, want = _operands(dev, dt, M, N, K)
    buf = torch.full((2, GUARD + M * N + GUARD + -M * N % 8), 7.0, dtype=dt, device=dev)   # both rows 16-byte aligned
    D, D2 = (b[GUARD:GUARD + M * N] for b in buf)
    c, ws, need = _call(0, dt, 1, A, B, D, deliver=D2.data_ptr())
    assert need > 4096                      # this shape is split
    for _ in range(2):
        D.fill_(7.0)
        D2.fill_(7.0)
        capi.check(capi.lib().fo_gemm_launch(C.byref(c), None))
        torch.cuda.synchronize()
        assert torch.equal(D.view(M, N), want) and torch.equal(D2.view(M, N), want)
    assert (buf[:, :GUARD] == 7.0).all() and (buf[:, GUARD + M * N:] == 7.0).all()
    assert not ws[:1024].any() and (ws[need // 4:] == 1e30).all()


@pytest.mark.parametrize("M,N,K", [(128, 128, 8192), (33, 129, 4104), (100, 1160, 7168), (128, 4096, 4096), (256, 2048, 4160)])
def test_split_plain_by_a_second_launch(dev, M, N, K):
    """The shapes that go to 64x64 tiles, which add their parts up themselves, in 128x128 ones: the reduction stores
    whole and ragged tiles, and delivers them."""
    L = capi.lib()
    try:
        capi.check(L.fo_tune(b"macro_tile", 128))
        c = capi.GemmCall(mode=0, dtype=capi.FO_BF16, algo=1, M=M, N=N, K=K, rLDN=1, nslices=1)
        need = C.c_size_t()
        capi.check(L.fo_gemm_workspace(C.byref(c), C.byref(need)))
        tiles = -(-M // 128) * -(-N // 128)
        assert need.value > 4096 and (need.value - 4096) % (tiles * 128 * 128 * 4) == 0
        for dt in (torch.float16, torch.bfloat16):
            test_split_plain(dev, dt, M, N, K)
    finally:
        capi.check(L.fo_tune(b"macro_tile", 0))


@pytest.mark.parametrize("M,N,K,algo", [(128, 1024, 4096, 1), (384, 640, 2056, 1), (512, 256, 4096, 2), (256, 640, 4096, 4),
                                        (4352, 4096, 1544, 1)])
@pytest.mark.parametrize("ws", [1, 4])
def test_split_signal_and_scatter(dev, M, N, K, algo, ws):
    """Half of the groups signalled, half delivered."""
    print(f"split {M}x{N}x{K} algo {algo} ws {ws}", flush=True)
    dt = torch.bfloat16
    BM, BN, _ = capi.algo_tile(algo)
    TM, TN = M // BM, N // BN
    T = TM * TN
    A, B, want = _operands(dev, dt, M, N, K)
    RA = tiling.reorder_indices(T, tiling.raster_hint(M, N, algo), dev)
    cseg = tiling.uniform_cseg(T, max(1, T // 6))
    start = [sum(cseg[:g]) for g in range(len(cseg))]
    half = len(cseg) // 2
    first = start[half]
    cs = torch.tensor(cseg, dtype=torch.int32, device=dev)
    st = torch.tensor(start, dtype=torch.int32, device=dev)
    table = torch.repeat_interleave(torch.arange(len(cseg), dtype=torch.int32, device=dev), cs.long()).int()
    mm = torch.zeros(len(cseg), dtype=torch.int32, device=dev)
    D = torch.full((M * N,), 7.0, dtype=dt, device=dev)
    D2 = torch.full((M * N,), 7.0, dtype=dt, device=dev)
    RE = tiling.generate_row_remap_array(M, N, BM, BN, cseg, ws, dev)
    more = dict(cseg_dev=cs.data_ptr(), G=len(cseg), group_table=table.data_ptr(), MM=mm.data_ptr(), RA=RA.data_ptr(),
                RE=RE.data_ptr(), deliver=D2.data_ptr(), deliver_from=first, nslices=ws, slice_count=ws,
                slice_stride=M * N // ws, group_start=st.data_ptr())
    c, wsp, need = _call(2 if ws > 1 else 1, dt, algo, A, B, D, **more)
    assert need > 4096
    for _ in range(2):
        mm.zero_()
        capi.check(capi.lib().fo_gemm_launch(C.byref(c), None))
        torch.cuda.synchronize()
        assert mm.cpu().tolist() == cseg[:half] + [0] * (len(cseg) - half)
    assert not wsp[:1024].any() and (wsp[need // 4:] == 1e30).all()
    tiles = torch.empty(T, BM, BN, dtype=dt, device=dev)                    # slot -> tile
    tiles[RA.long()] = want.view(TM, BM, TN, BN).permute(0, 2, 1, 3).reshape(T, BM, BN)
    rows = torch.empty(T * BM, BN, dtype=dt, device=dev)
    rows[RE.long() if ws > 1 else slice(None)] = tiles.view(T * BM, BN)
    assert torch.equal(D.view(-1, BN), rows)
    got = D2.view(ws, T * BM // ws, BN)
    for g, n in enumerate(cseg):
        r0, nr = start[g] * BM, n * BM
        for k in range(ws):
            mine = got[k, r0 // ws:(r0 + nr) // ws]
            if g < half:
                assert (mine == 7.0).all()
            else:
                assert torch.equal(mine, rows[r0 + k * nr // ws:r0 + (k + 1) * nr // ws])


@pytest.mark.parametrize("M,N,K", [(256, 128, 64), (384, 256, 72), (8, 136, 128), (600, 385, 200), (1536, 2048, 192),
                                   (384, 256, 264), (600, 385, 840), (256, 384, 1664), (256, 384, 3008), (512, 385, 3072),
                                   (1152, 2176, 3520), (2048, 2048, 4096)])
def test_tall_tile_gives_the_bits_of_the_square_one(dev, M, N, K):
    """The 256x128 macro tile on fewer panels than its ring holds, as many, one more and several turns of it, half
    and ragged tiles, and on as many as begin apart in K where a workspace is passed: without one the order of additions is the same."""
    L = capi.lib()
    g = torch.Generator().manual_seed(M + N + K)
    A, B = (torch.randn(r, K, generator=g).to(torch.bfloat16).to(dev) for r in (M, N))
    got = []
    try:
        for macro in (128, 256128):
            capi.check(L.fo_tune(b"macro_tile", macro))
            D = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=dev)
            capi.check(L.fo_gemm(capi.FO_BF16, 1, M, N, K, A.data_ptr(), B.data_ptr(), D.data_ptr(), None))
            torch.cuda.synchronize()
            got.append(D)
    finally:
        capi.check(L.fo_tune(b"macro_tile", 0))
    assert torch.equal(got[0], got[1])


@pytest.mark.parametrize("M,N,algo", [(512, 512, 1), (384, 640, 1), (512, 384, 4), (640, 512, 0)])
@pytest.mark.parametrize("ws", [1, 4])
def test_tall_tile_signals_and_places(dev, M, N, algo, ws):
    L = capi.lib()
    K, dt = 136, torch.float16
    BM, BN, _ = capi.algo_tile(algo)
    TM, TN = M // BM, N // BN
    A, B, want = _operands(dev, dt, M, N, K)
    cseg = tiling.uniform_cseg(TM * TN, 3)
    RA = torch.randperm(TM * TN, generator=torch.Generator().manual_seed(3)).int().to(dev)
    RE = tiling.generate_row_remap_array(M, N, BM, BN, cseg, ws, dev)
    cs = torch.tensor(cseg, dtype=torch.int32, device=dev)
    mm = torch.zeros(len(cseg), dtype=torch.int32, device=dev)
    D = torch.full((M * N // BN, BN), 7.0, dtype=dt, device=dev)
    c = capi.GemmCall(mode=2 if ws > 1 else 1, dtype=capi.dtype_code(dt), algo=algo, M=M, N=N, K=K, rLDN=1,
                      cseg_dev=cs.data_ptr(), G=len(cseg), A=A.data_ptr(), B=B.data_ptr(), D=D.data_ptr(),
                      MM=mm.data_ptr(), RA=RA.data_ptr(), RE=RE.data_ptr(), nslices=ws)
    try:
        capi.check(L.fo_tune(b"macro_tile", 256128))
        capi.check(L.fo_gemm_launch(C.byref(c), None))
        torch.cuda.synchronize()
    finally:
        capi.check(L.fo_tune(b"macro_tile", 0))
    assert mm.cpu().tolist() == cseg
    rows = torch.empty(TM * TN, BM, BN, dtype=dt, device=dev)
    rows[RA.long()] = want.view(TM, BM, TN, BN).permute(0, 2, 1, 3).reshape(TM * TN, BM, BN)
    out = torch.empty(TM * TN * BM, BN, dtype=dt, device=dev)
    out[RE.long() if ws > 1 else slice(None)] = rows.view(-1, BN)
    assert torch.equal(D, out)


@pytest.mark.parametrize("M,N,K,algo", [(128, 128, 64, 1), (256, 384, 72, 1), (256, 256, 200, 2), (512, 128, 136, 4)])
@pytest.mark.parametrize("ws", [1, 8])
def test_small_tile_delivers_into_larger_layout_tiles(dev, M, N, K, algo, ws):
    """Nothing signalled: the 64x64 macro tile, four or eight of which share a layout tile."""
    L, dt = capi.lib(), torch.bfloat16
    BM, BN, _ = capi.algo_tile(algo)
    TM, TN = M // BM, N // BN
    T = TM * TN
    A, B, want = _operands(dev, dt, M, N, K)
    RA = torch.randperm(T, generator=torch.Generator().manual_seed(3)).int().to(dev)
    RE = tiling.generate_row_remap_array(M, N, BM, BN, [T], ws, dev)
    cs, zero = torch.tensor([T], dtype=torch.int32, device=dev), torch.zeros(T, dtype=torch.int32, device=dev)
    D, D2 = (torch.full((T * BM, BN), 7.0, dtype=dt, device=dev) for _ in range(2))
    mm = torch.zeros(1, dtype=torch.int32, device=dev)
    c = capi.GemmCall(mode=2 if ws > 1 else 1, dtype=capi.dtype_code(dt), algo=algo, M=M, N=N, K=K, rLDN=1,
                      cseg_dev=cs.data_ptr(), G=1, group_table=zero.data_ptr(), A=A.data_ptr(), B=B.data_ptr(),
                      D=D.data_ptr(), MM=mm.data_ptr(), RA=RA.data_ptr(), RE=RE.data_ptr(), nslices=ws, slice_count=ws,
                      slice_stride=M * N // ws, group_start=zero.data_ptr(), deliver=D2.data_ptr())
    capi.check(L.fo_gemm_launch(C.byref(c), None))
    torch.cuda.synchronize()
    rows = torch.empty(T, BM, BN, dtype=dt, device=dev)
    rows[RA.long()] = want.view(TM, BM, TN, BN).permute(0, 2, 1, 3).reshape(T, BM, BN)
    out = torch.empty(T * BM, BN, dtype=dt, device=dev)
    out[RE.long() if ws > 1 else slice(None)] = rows.view(-1, BN)
    assert torch.equal(D, out) and torch.equal(D2, out) and mm.item() == 0


def test_timed_call_runs_what_the_untimed_one_does(dev):
    """The event pair of fo_time_next_launch spans both launches of a split call, and leaves the call as it is."""
    L, dt, (M, N, K) = capi.lib(), torch.bfloat16, (128, 4096, 7168)
    g = torch.Generator().manual_seed(5)
    A, B = (torch.randn(r, K, generator=g).to(dt).to(dev) for r in (M, N))
    evs = [C.c_void_p() for _ in range(4)]
    for e in evs:
        capi.check(L.fo_event_create(C.byref(e)))
    inner0, inner1, outer0, outer1 = evs
    got = []
    for timed, split in ((False, False), (False, True), (True, True)):
        D = torch.zeros(M, N, dtype=dt, device=dev)
        c, ws, need = _call(0, dt, 1, A, B, D)
        assert need > 4096
        if not split:
            c.workspace, c.workspace_bytes = None, 0
        torch.cuda.synchronize()
        capi.check(L.fo_event_record(outer0, None))
        if timed:
            capi.check(L.fo_time_next_launch(inner0, inner1))
        capi.check(L.fo_gemm_launch(C.byref(c), None))
        capi.check(L.fo_event_record(outer1, None))
        torch.cuda.synchronize()
        got.append(D)
    assert not torch.equal(got[0], got[1])      # the order of additions shows which of the two ran
    assert torch.equal(got[1], got[2])
    inner, outer = C.c_float(), C.c_float()
    capi.check(L.fo_event_elapsed_ms(inner0, inner1, C.byref(inner)))
    capi.check(L.fo_event_elapsed_ms(outer0, outer1, C.byref(outer)))
    for e in evs:
        capi.check(L.fo_event_destroy(e))
    assert 0 < inner.value <= outer.value
    assert 2 * (M + N) * K / (inner.value * 1e-3) < 10e12    # the operands' bytes alone: the first launch is in it
