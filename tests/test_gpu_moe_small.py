"""The one-launch index build at the edges of its range, the combine's column
split, and the expert GEMMs' tile order from padded counts and from rb_expert."""
import numpy as np
import pytest
import torch

from mkernel_amd import ops, workloads as wl

pytestmark = pytest.mark.gpu

TABLES = ("padded_tokens_per_expert", "local_rb_per_expert", "pull_indices", "row_expert", "rb_expert", "rb_rows",
          "row_weight", "owner_offset", "row_to_slot", "row_to_owner", "slot_to_row")


# around the small build's limits: 4096 entries, 1024 tokens, 256 experts
@pytest.mark.parametrize("T,k,experts,e0,n_local,block", [
    (1, 1, 8, 0, 8, 128), (1, 8, 256, 0, 32, 128), (64, 8, 256, 32, 32, 128), (127, 8, 64, 8, 16, 128),
    (128, 8, 16, 0, 16, 64), (129, 8, 40, 3, 17, 128), (512, 8, 256, 0, 256, 128), (513, 8, 256, 0, 256, 128),
    (512, 8, 300, 0, 257, 128), (1024, 4, 32, 0, 32, 128), (1025, 3, 32, 0, 32, 128), (455, 9, 24, 0, 24, 1),
    (4, 1024, 64, 0, 64, 128), (333, 2, 2, 1, 1, 128)])
def test_index_small_build(dev, T, k, experts, e0, n_local, block):
    print(f"index small T={T} k={k} experts={experts} e0={e0} n_local={n_local} block={block}", flush=True)
    rng = np.random.default_rng(T * 31 + k)
    for ids in (rng.integers(0, experts, size=(T, k)), np.full((T, k), e0)):
        ids, gates = ids.astype(np.int32), rng.random((T, k), dtype=np.float32)
        host = ops.moe_build_indices(ids, gates, e0, n_local, block)
        gpu = ops.moe_build_indices_dev(torch.from_numpy(ids).to(dev), torch.from_numpy(gates).to(dev), e0, n_local,
                                        block)
        assert (gpu["R"], gpu["R_pad"]) == (host["R"], host["R_pad"])
        for f in TABLES:
            assert np.array_equal(gpu[f].cpu().numpy(), np.asarray(host[f])), f


@pytest.mark.parametrize("out", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,H,k", [(1, 7168, 8), (3, 8, 2), (7, 2056, 8), (200, 1032, 3), (1500, 512, 8), (5, 4096, 20)])
def test_combine_sizes(dev, T, H, k, out):
    print(f"combine T={T} H={H} k={k} out={out}", flush=True)
    rng = np.random.default_rng(T + H + k)
    ids = np.stack([rng.permutation(32)[:k] for _ in range(T)]).astype(np.int32)
    gates = rng.random((T, k), dtype=np.float32)
    d = ops.moe_build_indices_dev(torch.from_numpy(ids).to(dev), torch.from_numpy(gates).to(dev), 0, 24)
    ye = wl.randn_bf16((max(d["R_pad"], 1), H), 5).to(dev)
    y = torch.full((T, H), float("nan"), dtype=out, device=dev)
    ops.moe_combine(ye, d["row_weight"], d["owner_offset"], d["slot_to_row"], y)
    ref = torch.zeros((T, H), dtype=torch.float64)
    pull, w, rows = d["pull_indices"].cpu(), d["row_weight"].cpu().double(), ye.cpu().double()
    for r in range(d["R_pad"]):
        if pull[r, 0] >= 0:
            ref[pull[r, 2]] += w[r] * rows[r]
    # k fp32 products and sums of magnitude below 8 each; bf16 rounds once more
    atol = 20 * 8 * 2.0 ** -23
    rtol = 2 ** -8 if out is torch.bfloat16 else 0
    assert torch.allclose(y.cpu().double(), ref, rtol=rtol, atol=atol)


@pytest.mark.parametrize("counts", [[130, 0, 1, 700, 5], [0, 0, 9, 0, 0], [128] * 5, [1, 1, 1, 1, 1500]])
@pytest.mark.parametrize("K,Nw,mode", [(256, 512, 0), (288, 4608, 0), (4128, 1024, 1), (4096, 768, 0)])
def test_grouped_gemm_orders(dev, counts, K, Nw, mode):
    """The same tiles whichever table names the experts, and every row right."""
    print(f"grouped counts={counts} K={K} Nw={Nw} mode={mode}", flush=True)
    padded = [(c + 127) // 128 * 128 for c in counts]
    R, E = sum(padded), len(counts)
    A = wl.randn_bf16((R, K), 1, K ** -0.5).to(dev)
    W = wl.randn_bf16((E, K, Nw), 2, K ** -0.5).to(dev)
    rb_expert = torch.tensor([e for e in range(E) for _ in range(padded[e] // 128)], dtype=torch.int32, device=dev)
    ppe = torch.tensor(padded, dtype=torch.int32, device=dev)
    width = Nw // 2 if mode else Nw
    outs = []
    for kw in ({"rb_expert": rb_expert}, {"padded_tokens_per_expert": ppe},
               {"rb_expert": rb_expert, "sizes": torch.tensor([R, R], dtype=torch.int64, device=dev)}):
        out = torch.full((R, width), float("nan"), dtype=torch.bfloat16, device=dev)
        ops.moe_grouped_gemm(A, W, out, mode=mode, **kw)
        outs.append(out)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    row = 0
    for e in range(E):
        h = A[row:row + padded[e]].float().cpu() @ W[e].float().cpu()
        if mode:
            h = torch.nn.functional.silu(h[:, :width]) * h[:, width:]
        got = outs[0][row:row + padded[e]].float().cpu()
        # one bf16 rounding of fp32 sums in another order (and of HIP's fast exponential)
        assert torch.allclose(got, h, rtol=2 ** -7, atol=1e-4), e
        row += padded[e]


@pytest.mark.parametrize("counts,rows", [([256, 512, 128], 512), ([256, 256, 128], 384), ([128, 384, 0, 640], 896),
                                         ([64, 448, 512], 384), ([128, 128], 512)])
@pytest.mark.parametrize("K,Nw,mode", [(288, 1024, 0), (256, 768, 1), (4128, 512, 0)])
def test_grouped_gemm_counts_past_the_rows(dev, counts, rows, K, Nw, mode):
    """Padded counts that do not sum to the launch's rows (a table built for
    more rows than the buffers hold, or one that ends before them): every row of
    the launch is right, and nothing behind the output is written."""
    print(f"grouped counts={counts} rows={rows} K={K} Nw={Nw} mode={mode}", flush=True)
    E, width, guard = len(counts), Nw // 2 if mode else Nw, 1024
    A = wl.randn_bf16((rows + guard, K), 1, K ** -0.5).to(dev)
    W = wl.randn_bf16((E, K, Nw), 2, K ** -0.5).to(dev)
    ppe = torch.tensor(counts, dtype=torch.int32, device=dev)
    rb_rows = torch.full(((rows + guard) // 128,), 128, dtype=torch.int32, device=dev)
    total = sum(counts)
    outs = []
    for kw in ({}, {"rb_rows": rb_rows}, {"sizes": torch.tensor([total, max(total, rows)], dtype=torch.int64, device=dev)}):
        out = torch.full((rows + guard, width), 7.0, dtype=torch.bfloat16, device=dev)
        ops.moe_grouped_gemm(A[:rows], W, out[:rows], mode=mode, padded_tokens_per_expert=ppe, **kw)
        torch.cuda.synchronize()
        assert bool((out[rows:] == 7.0).all()), "written past the launch's rows"
        outs.append(out[:rows])
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    ends = np.cumsum(counts)
    for r in range(0, rows, 128):  # a row tile belongs to the expert of its first row
        e = min(int(np.searchsorted(ends, r, side="right")), E - 1)
        h = A[r:r + 128].float().cpu() @ W[e].float().cpu()
        if mode:
            h = torch.nn.functional.silu(h[:, :width]) * h[:, width:]
        # one bf16 rounding of fp32 sums in another order (and of HIP's fast exponential)
        assert torch.allclose(outs[0][r:r + 128].float().cpu(), h, rtol=2 ** -7, atol=1e-4), r


@pytest.mark.parametrize("blocks", [16, 12, 11, 10, 3, 0])
@pytest.mark.parametrize("mode", [0, 1])
def test_tile_width_follows_the_device_rows(dev, blocks, mode):
    """With a device row count the tile width follows the row blocks that are
    there, however tight the capacity: bit-equal to the wide tiles above 10
    blocks, to the narrow ones up to 10.  (K is split differently there.)"""
    print(f"tile width blocks={blocks} mode={mode}", flush=True)
    E, K, Nw = 16, 4128, 4096
    g = torch.Generator(device=dev).manual_seed(blocks)
    A = torch.randn((E * 128, K), generator=g, device=dev).mul_(K ** -0.5).to(torch.bfloat16)
    W = torch.empty((E, K, Nw), dtype=torch.bfloat16, device=dev)
    for e in range(E):
        W[e] = torch.randn((K, Nw), generator=g, device=dev).mul_(K ** -0.5)
    rb = torch.arange(E, dtype=torch.int32, device=dev)
    sizes = torch.tensor([blocks * 128, blocks * 128], dtype=torch.int64, device=dev)
    width = Nw // 2 if mode else Nw
    outs = {}
    for tile_n in (0, 256, 512):
        for ws in (None, False):
            out = torch.full((E * 128, width), 7.0, dtype=torch.bfloat16, device=dev)
            ops.moe_grouped_gemm(A, W, out, rb_expert=rb, mode=mode, sizes=sizes, tile_n=tile_n, split_ws=ws)
            torch.cuda.synchronize()
            assert bool((out[blocks * 128:] == 7.0).all())
            outs[tile_n, ws] = out
    assert torch.equal(outs[0, None], outs[256 if blocks <= 10 else 512, None])
    if blocks >= 10:
        assert not torch.equal(outs[256, None], outs[512, None]), "the widths are told apart by their K-split"
    for b in range(blocks):
        h = A[b * 128:(b + 1) * 128].float() @ W[b].float()
        if mode:
            h = torch.nn.functional.silu(h[:, :width]) * h[:, width:]
        # one bf16 rounding of fp32 sums in another order (and of HIP's fast exponential)
        for out in (outs[0, None], outs[0, False]):
            assert torch.allclose(out[b * 128:(b + 1) * 128].float(), h, rtol=2 ** -7, atol=1e-4), b
