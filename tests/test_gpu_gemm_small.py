"""The small-tile GEMM: edges
of its tiles and K stages, K-split parts, strides, and what lies around the
operands."""
import numpy as np
import pytest
import torch

from mkernel_amd import capi, ops, workloads as wl
from mkernel_amd.capi import GemmArgs
from oracle.gemm import gemm_ref, rel_fro

pytestmark = pytest.mark.gpu

# one 64 x 64 tile row to a full round, each tile shape, one and several parts
# per tile, K of one half stage, of an odd number of half stages, and long
SHAPES = [(128, 256, 32), (128, 256, 96), (128, 2048, 2048), (640, 512, 4128), (512, 512, 4096), (2048, 1024, 224),
          (2048, 1024, 2048), (1024, 2048, 992), (512, 2048, 8192), (2048, 2048, 1024), (1920, 2816, 608),
          (384, 3584, 5280), (1664, 2560, 416), (4224, 2304, 288), (512, 2816, 5984), (4480, 3584, 96),
          (1280, 1792, 5152)]


def _call(A, B, C, M, N, K, lda, ldb, ldc, ws):
    capi.call("mk_gemm", GemmArgs(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, lda, ldb, ldc, 0, 0, 0,
                                  ws.data_ptr() if ws is not None else None, ws.numel() if ws is not None else 0),
              torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_small_gemm_vs_oracle(dev, M, N, K):
    print(f"small gemm M={M} N={N} K={K}", flush=True)
    A, B = wl.randn_bf16((M, K), 1, K ** -0.5), wl.randn_bf16((K, N), 2, K ** -0.5)
    ref = gemm_ref(A, B)
    ws = torch.zeros(int(capi.lib().mk_query_workspace_bytes(0, M, N, K)), dtype=torch.uint8, device=dev)
    Ad, Bd = A.to(dev), B.to(dev)
    outs = []
    for _ in range(3):
        C = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)
        _call(Ad, Bd, C, M, N, K, K, N, N, ws)
        torch.cuda.synchronize()
        outs.append(C)
        assert int(ws[:4096].view(torch.int32).abs().sum()) == 0, "workspace words not left zero"
    # one bf16 rounding (2^-8 of the value) of an fp32 sum taken in another order
    assert torch.allclose(outs[0].cpu().float(), ref, rtol=2 ** -7, atol=1e-5)
    assert all(torch.equal(outs[0], o) for o in outs[1:]), "not deterministic"
    whole = ops.gemm(Ad, Bd, split_ws=False)  # no workspace: every tile whole
    assert torch.allclose(whole.cpu().float(), ref, rtol=2 ** -7, atol=1e-5)


@pytest.mark.parametrize("M,N,K", [(128, 512, 96), (512, 512, 4128), (2048, 1024, 160), (1920, 768, 32)])
def test_small_gemm_strides_and_surroundings(dev, M, N, K):
    """Padded rows: what lies between the rows of A, B (NaN) is not read into
    the result, what lies between the rows of C is not written."""
    lda, ldb, ldc = K + 40, N + 24, N + 8
    A, B = wl.randn_bf16((M, K), 3, K ** -0.5), wl.randn_bf16((K, N), 4, K ** -0.5)
    Ad = torch.full((M, lda), float("nan"), dtype=torch.bfloat16, device=dev)
    Bd = torch.full((K, ldb), float("nan"), dtype=torch.bfloat16, device=dev)
    C = torch.full((M, ldc), 7.0, dtype=torch.bfloat16, device=dev)
    Ad[:, :K], Bd[:, :N] = A.to(dev), B.to(dev)
    _call(Ad, Bd, C, M, N, K, lda, ldb, ldc, ops.split_workspace())
    torch.cuda.synchronize()
    assert torch.allclose(C[:, :N].cpu().float(), gemm_ref(A, B), rtol=2 ** -7, atol=1e-5)
    assert bool((C[:, N:] == 7.0).all())


def test_small_gemm_row_infinities_stay_in_their_row(dev):
    """K ends inside a stage: the row after it holds infinities and NaN, which
    must reach its own outputs only."""
    M, N, K = 256, 512, 160
    A, B = wl.randn_bf16((M, K), 5), wl.randn_bf16((K, N), 6, K ** -0.5)
    A[1], A[77] = float("inf"), float("nan")
    C = ops.gemm(A.to(dev), B.to(dev)).cpu().float()
    ok = torch.ones(M, dtype=torch.bool)
    ok[[1, 77]] = False
    assert torch.isfinite(C[ok]).all() and not torch.isfinite(C[~ok]).any()
    assert torch.allclose(C[ok], gemm_ref(A[ok], B), rtol=2 ** -7, atol=1e-3)


def test_small_gemm_on_several_streams(dev):
    """K-split launches on four streams at once, each with its own workspace."""
    M, N, K = 512, 1024, 8192
    streams = [torch.cuda.Stream() for _ in range(4)]
    A = [wl.randn_bf16((M, K), 10 + i, K ** -0.5).to(dev) for i in range(4)]
    B = [wl.randn_bf16((K, N), 20 + i, K ** -0.5).to(dev) for i in range(4)]
    want = [ops.gemm(a, b).clone() for a, b in zip(A, B)]
    C = [torch.empty((M, N), dtype=torch.bfloat16, device=dev) for _ in range(4)]
    torch.cuda.synchronize()
    for _ in range(10):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                ops.gemm(A[i], B[i], C[i])
    torch.cuda.synchronize()
    assert all(torch.equal(c, w) for c, w in zip(C, want))
    assert rel_fro(C[0].float(), gemm_ref(A[0].cpu(), B[0].cpu())) < 2e-2


@pytest.mark.parametrize("M,N,K", [(640, 512, 4128), (512, 512, 4096), (1024, 512, 8192), (512, 2048, 8192)])
def test_small_gemm_beside_flags_of_a_launch_that_gave_up(dev, M, N, K):
    """K-split flags that a gated launch left set when its bounded wait gave up
    (any of the words the persistent kernel uses) do not reach the small
    kernel's own words."""
    print(f"small gemm, set split flags, M={M} N={N} K={K}", flush=True)
    A, B = wl.randn_bf16((M, K), 1, K ** -0.5).to(dev), wl.randn_bf16((K, N), 2, K ** -0.5).to(dev)
    ws = torch.zeros(int(capi.lib().mk_query_workspace_bytes(0, M, N, K)), dtype=torch.uint8, device=dev)
    want, C = (torch.empty((M, N), dtype=torch.bfloat16, device=dev) for _ in range(2))
    _call(A, B, want, M, N, K, K, N, N, ws)
    torch.cuda.synchronize()
    assert bool((ws[4096:].view(torch.int32) != 0).any()), "no tile was split along K"
    words = ws[:2048].view(torch.int32)
    words.fill_(1)
    for _ in range(2):
        C.zero_()
        _call(A, B, C, M, N, K, K, N, N, ws)
        torch.cuda.synchronize()
        assert torch.equal(C, want) and bool((words == 1).all()) and not bool(ws[2048:4096].any())
