"""AllGather / ReduceScatter / AllReduce launches that stage first and then run
the small-tile kernel, against the persistent kernel (the same call with the
grid named) and the oracle: bit-equal outputs, staged bytes, flags."""
import ctypes

import numpy as np
import pytest
import torch

from mkernel_amd import capi, ops, workloads as wl
from oracle.gemm import gemm_ref

pytestmark = pytest.mark.gpu

# every tile shape that each operation may get, and blocks staged first before
# the persistent kernel (the last of AG and of RS); tests/test_plans.py says so
AG = [(2, 512, 256, 32, 0), (16, 4096, 256, 1056, 2), (4, 2048, 512, 992, 4), (8, 4096, 1024, 512, 0),
      (1, 256, 768, 96, 2), (3, 768, 512, 4128, 0), (2, 1536, 2816, 288, 3), (2, 3584, 1792, 160, 0),
      (4, 7168, 1792, 32, 0), (4, 5120, 3328, 32, 1), (16, 20480, 1536, 32, 0)]
RS = [(2, 1, 512, 256, 32), (16, 5, 4096, 4096, 256), (4, 0, 2048, 768, 416), (1, 0, 512, 512, 96),
      (8, 7, 2048, 1024, 2080), (2, 0, 1536, 2304, 160), (8, 3, 2048, 256, 32), (4, 2, 5120, 3328, 32),
      (2, 1, 3584, 1792, 160), (8, 0, 10240, 1280, 32), (8, 6, 6144, 256, 32), (2, 1, 2560, 3584, 32)]
AR = [(4, 512, 512, 64), (8, 2048, 1024, 992), (2, 2560, 768, 160), (2, 512, 256, 288)]
AR2 = [(4, 2, 2048, 512, 96), (2, 0, 1024, 1024, 544), (8, 7, 2048, 2304, 32)]
DONE = [(4, 512, 512, 64, False), (8, 2048, 1024, 992, False), (2, 2560, 768, 160, False), (2, 512, 256, 288, False),
        (2, 3584, 1792, 160, False), (4, 5120, 3328, 32, False), (4, 6144, 3584, 32, False), (2, 1536, 2816, 32, False),
        (16, 4096, 4096, 256, True), (8, 2048, 2304, 32, True), (2, 1024, 1024, 544, True), (8, 10240, 1280, 32, True)]


def _words(n, dev):
    return torch.zeros(n, dtype=torch.int32, device=dev)


def _perm(n, dev, seed):
    return torch.from_numpy(np.random.default_rng(seed).permutation(n).astype(np.int32)).to(dev)


@pytest.mark.parametrize("producers", [-1, -2])
@pytest.mark.parametrize("world,M,N,K,present", AG)
def test_ag_small(dev, world, M, N, K, present, producers):
    print(f"ag small world={world} M={M} N={N} K={K} present={present} producers={producers}", flush=True)
    A, B = wl.randn_bf16((M, K), 1, K ** -0.5), wl.randn_bf16((K, N), 2, K ** -0.5)
    Ad, Bd, n = A.to(dev), B.to(dev), M // 128
    order = _perm(n, dev, 3)
    outs = []
    for cus in (0, ops.cu_count()):
        full = torch.zeros_like(Ad)
        for b in order[:present].tolist():
            full[b * 128:(b + 1) * 128] = Ad[b * 128:(b + 1) * 128]
        flags, counters = _words(n, dev), _words(n, dev)
        C = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)
        for epoch in (1, 2):
            ops.ag_gemm(Ad, full, Bd, C, flags, order, epoch=epoch, num_producers=producers, num_cus=cus,
                        stage_counters=counters, n_present=present)
        torch.cuda.synchronize()
        assert torch.equal(full, Ad) and bool((flags == 2).all())
        outs.append(C)
    plain = ops.ag_gemm(None, Ad, Bd, torch.empty_like(C), None, None, epoch=1, gated=False, num_producers=0)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], plain)
    # one bf16 rounding (2^-8 of the value) of an fp32 sum taken in another order
    assert torch.allclose(outs[0].cpu().float(), gemm_ref(A, B), rtol=2 ** -7, atol=1e-5)


@pytest.mark.parametrize("world,rank,M,N,K", RS)
def test_rs_small(dev, world, rank, M, N, K):
    print(f"rs small world={world} rank={rank} M={M} N={N} K={K}", flush=True)
    A, B = wl.randn_bf16((M, K), 4, K ** -0.5), wl.randn_bf16((K, N), 5, K ** -0.5)
    Ad, Bd, rows = A.to(dev), B.to(dev), M // world
    peers = wl.randn_bf16((world - 1, rows, N), 6, 0.5).to(dev)
    n = (world - 1) * rows // 128
    order = _perm(n, dev, 7) if n else None
    outs = []
    for cus in (0, ops.cu_count()):
        flags, counters = _words(max(n, 1), dev), _words(max(n, 1), dev)
        recv, sends = torch.zeros_like(peers), torch.full((M, N), 3.0, dtype=torch.bfloat16, device=dev)
        out = torch.empty((rows, N), dtype=torch.bfloat16, device=dev)
        ops.gemm_rs(Ad, Bd, sends, out, peers if n else None, recv if n else None, world, rank, flags, order, epoch=5,
                    num_cus=cus, stage_counters=counters)
        torch.cuda.synchronize()
        assert torch.equal(recv, peers) and (n == 0 or bool((flags == 5).all()))
        assert bool((sends[rank * rows:(rank + 1) * rows] == 3.0).all()), "own rows are not sent"
        outs.append((out, sends))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    ref = gemm_ref(A, B)
    own = ref[rank * rows:(rank + 1) * rows] + peers.cpu().float().sum(0)
    # the fold's fp32 sum in another order, then one bf16 rounding
    assert torch.allclose(outs[0][0].cpu().float(), own, rtol=2 ** -7, atol=1e-5)


@pytest.mark.parametrize("world,M,N,K", AR)
def test_ar_small(dev, world, M, N, K):
    print(f"ar small world={world} M={M} N={N} K={K}", flush=True)
    A, B = wl.randn_bf16((M, K), 8, K ** -0.5).to(dev), wl.randn_bf16((K, N), 9, K ** -0.5).to(dev)
    peers = wl.randn_bf16((world - 1, M, N), 10, 0.5).to(dev)
    n = (world - 1) * M // 128
    epoch = torch.full((1,), 6, dtype=torch.int32, device=dev)
    outs = []
    for cus in (0, ops.cu_count()):
        flags, counters, done = _words(n, dev), _words(n, dev), _words((M // 256) * (N // 256), dev)
        recv, C = torch.zeros_like(peers), torch.empty((M, N), dtype=torch.bfloat16, device=dev)
        ops.gemm_ar(A, B, C, peers, recv, world, flags, _perm(n, dev, 11), epoch=1, num_cus=cus,
                    stage_counters=counters, done_flags=done, epoch_ptr=epoch)
        torch.cuda.synchronize()
        assert torch.equal(recv, peers) and bool((flags == 6).all()) and bool((done == 6).all())
        outs.append(C)
    assert torch.equal(outs[0], outs[1])
    ref = gemm_ref(A.cpu(), B.cpu()) + peers.cpu().float().sum(0)
    assert torch.allclose(outs[0].cpu().float(), ref, rtol=2 ** -7, atol=1e-5)


@pytest.mark.parametrize("world,rank,M,N,K", AR2)
def test_ar_two_shot_small(dev, world, rank, M, N, K):
    print(f"ar two-shot small world={world} rank={rank} M={M} N={N} K={K}", flush=True)
    A, B = wl.randn_bf16((M, K), 13, K ** -0.5).to(dev), wl.randn_bf16((K, N), 14, K ** -0.5).to(dev)
    s = M // world
    peers, reduced = (wl.randn_bf16((world - 1, s, N), seed, 0.5).to(dev) for seed in (15, 16))
    n = 2 * (world - 1) * s // 128
    flags, counters, done = _words(n, dev), _words(n, dev), _words((M // 256) * (N // 256), dev)
    C, sends = (torch.full((M, N), 3.0, dtype=torch.bfloat16, device=dev) for _ in range(2))
    recv = torch.zeros_like(peers)
    ops.gemm_ar_two_shot(A, B, C, sends, peers, recv, reduced, world, rank, flags, _perm(n, dev, 17), epoch=9,
                         stage_counters=counters, done_flags=done)
    torch.cuda.synchronize()
    ref = gemm_ref(A.cpu(), B.cpu())
    lo, hi = rank * s, (rank + 1) * s
    assert torch.allclose(C[lo:hi].cpu().float(), ref[lo:hi] + peers.cpu().float().sum(0), rtol=2 ** -7, atol=1e-5)
    assert torch.equal(torch.cat([C[:lo], C[hi:]]).view(world - 1, s, N), reduced) and torch.equal(recv, peers)
    sent = torch.ones(M, dtype=torch.bool)
    sent[lo:hi] = False
    assert torch.allclose(sends[sent.to(dev)].cpu().float(), ref[sent], rtol=2 ** -7, atol=1e-5)
    assert bool((sends[lo:hi] == 3.0).all()) and bool((flags == 9).all())
    per = N // 256
    assert bool((done[lo // 256 * per:hi // 256 * per] == 9).all())
    assert int((done != 0).sum()) == s // 256 * per


@pytest.mark.parametrize("world,M,N,K,two_shot", DONE)
def test_done_flags_come_from_the_tiles(dev, world, M, N, K, two_shot):
    """Done flags are published by the launch that folds the tiles, not by one
    behind it, under several epochs (the parts are counted in the workspace,
    which is left zeroed), and without a workspace, or with one too small for
    its words, too: then nothing behind it is touched."""
    print(f"done flags world={world} M={M} N={N} K={K} two_shot={two_shot}", flush=True)
    A, B = wl.randn_bf16((M, K), 8, K ** -0.5).to(dev), wl.randn_bf16((K, N), 9, K ** -0.5).to(dev)
    rows, rank = (M // world, world - 1) if two_shot else (M, 0)
    peers = wl.randn_bf16((world - 1, rows, N), 10, 0.5).to(dev)
    reduced = wl.randn_bf16((world - 1, rows, N), 11, 0.5).to(dev)
    n = (world - 1) * rows // 128 * (1 + two_shot)
    ws = torch.zeros(int(capi.lib().mk_query_workspace_bytes(0, M, N, K)), dtype=torch.uint8, device=dev)
    flags, counters, done = _words(n, dev), _words(n, dev), _words((M // 256) * (N // 256), dev)
    recv = torch.zeros_like(peers)
    C, sends = (torch.empty((M, N), dtype=torch.bfloat16, device=dev) for _ in range(2))
    epoch = torch.full((1,), 3, dtype=torch.int32, device=dev)

    def call(ws, done, **kw):
        if two_shot:
            ops.gemm_ar_two_shot(A, B, C, sends, peers, recv, reduced, world, rank, flags, None, epoch=1,
                                 stage_counters=counters, done_flags=done, split_ws=ws, **kw)
        else:
            ops.gemm_ar(A, B, C, peers, recv, world, flags, None, epoch=1, stage_counters=counters, done_flags=done,
                        split_ws=ws, **kw)

    lo, hi = rank * rows // 256 * (N // 256), (rank + 1) * rows // 256 * (N // 256)
    outs = []
    little = torch.full((4096,), 7, dtype=torch.uint8, device=dev)
    for split in (ws, ws, False, little[:1024]):
        epoch += 1
        done.zero_()
        call(split, done, epoch_ptr=epoch)
        torch.cuda.synchronize()
        assert bool((done[lo:hi] == epoch).all()) and int((done != 0).sum()) == hi - lo
        assert not bool(ws[:4096].any()) and bool((little == 7).all())
        outs.append(C.clone())
    assert all(torch.equal(outs[0], o) for o in outs[1:])
    assert _graph_nodes(lambda: call(ws, done, epoch_ptr=epoch)) == _graph_nodes(lambda: call(ws, None, epoch_ptr=epoch))


def _graph_nodes(call):
    """Nodes of the graph that `call` is captured into."""
    g = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(g):
        call()
    n = ctypes.c_size_t(0)
    hip = ctypes.CDLL("libamdhip64.so")
    assert hip.hipGraphGetNodes(ctypes.c_void_p(g.raw_cuda_graph()), None, ctypes.byref(n)) == 0
    return n.value
