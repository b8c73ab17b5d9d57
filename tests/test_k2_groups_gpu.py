"""K2 attention at the edges of its work items: four query heads per KV head (24 groups of 16 rows
over 8 waves), chunks of at most half an item's queries (the waves of a pair take half of every
tile's keys each), and last blocks of one query, against the CPU oracle."""
import pytest
import torch

from helpers import dec_pool_of, fitted_store, llama3_cache, paged
from oracle import attend, rope
from vllm_ttkv import kernels, synth

pytestmark = pytest.mark.gpu
SCALE = 128 ** -0.5


@pytest.mark.parametrize("cfg,H,G,r1,dtype,lens,qlens", [
    ("safe", 8, 4, 110, torch.float16, [700, 333, 65], [49, 48, 64]),   # one past half, half
    ("campaign4x", 8, 4, 110, torch.bfloat16, [900, 97], [97, 96]),     # one past an item
    ("safe", 4, 4, 64, torch.float16, [1500], [2]),
    ("tight", 8, 4, 128, torch.float16, [400, 401, 402], [17, 1, 200]),
    ("safe", 8, 3, 110, torch.float16, [700, 640, 64], [65, 64, 16]),   # one past half, half
    ("campaign4x", 8, 3, 96, torch.float16, [515, 130], [129, 19]),
    ("safe", 8, 3, 110, torch.float16, [3000], [5]),                    # many key splits
    ("safe", 8, 2, 110, torch.float16, [300, 200], [33, 128]),
    ("safe", 2, 1, 110, torch.bfloat16, [300, 70], [64, 70]),           # a whole context
])
def test_row_groups(cfg, H, G, r1, dtype, lens, qlens):
    print(f"[k2 groups] {cfg} H={H} G={G} r1={r1} {lens} {qlens}", flush=True)
    stores = [fitted_store(cfg, n, seed=40 + i, r1=r1, H_=H) for i, n in enumerate(lens)]
    pg = paged(stores, 16, 3)
    lay = stores[0]["lay"]
    q = synth.queries(sum(qlens), HQ=H * G, seed=9, dtype=dtype)
    qsl = torch.tensor([0] + list(torch.tensor(qlens).cumsum(0)), dtype=torch.int32)
    cache = llama3_cache(4096)
    dev = "cuda"
    dec_map = torch.full((pg["num_blocks"],), -1, dtype=torch.int32)
    for r in range(len(lens)):
        dec_map[pg["block_table"][r, 0]] = r
    out = torch.full((sum(qlens), H * G, 128), float("nan"), dtype=dtype, device=dev)
    err = torch.zeros(1, dtype=torch.int32, device=dev)
    ws = kernels.prefill_workspace(lay, H * G, len(lens), max(qlens), max(lens), dev)
    args = (lay, q.to(dev), pg["page"].to(dev), 16, pg["block_table"].to(dev),
            pg["seq_lens"].to(dev), qsl.to(dev), max(qlens), max(lens), dec_map.to(dev),
            dec_pool_of([s["decoder"] for s in stores], dev), cache.to(dev), SCALE)
    kernels.prefill_paged(*args, out=out, workspace=ws, error_word=err)
    torch.cuda.synchronize()
    assert int(err.item()) == 0
    first = out.float().cpu()
    kernels.prefill_paged(*args, out=out.fill_(0), workspace=ws, error_word=err)
    assert torch.equal(out.float().cpu(), first)        # the counters came back to zero
    want = attend.paged_continuation(lay, pg["page"], pg["block_table"], pg["seq_lens"], qsl,
                                     q.float(), [s["decoder"] for s in stores], cache, 16, SCALE,
                                     dtype=torch.float64)
    tol = 1.0 if dtype == torch.float16 else 8.0        # bf16 rounds the output 8 times coarser
    for r in range(len(lens)):
        e = (first[qsl[r]:qsl[r + 1]].double() - want[r]).abs()
        assert e.max() <= tol * 2e-3 and e.mean() <= tol * 1e-3, (r, e.max(), e.mean())


@pytest.mark.parametrize("G,n,Q", [(4, 300, 40), (4, 300, 130), (3, 300, 40), (3, 300, 130),
                                   (1, 200, 70)])
@pytest.mark.parametrize("scale", [-0.09, 0.0])
def test_scales_that_are_not_positive(G, n, Q, scale):
    """A negative scale turns the order of the scores and a zero one makes them alike; the keys
    past a query stay hidden under both."""
    print(f"[k2 scale] G={G} n={n} Q={Q} scale={scale}", flush=True)
    st = fitted_store("safe", n, seed=60)
    pg = paged([st], 16, 4)
    q = synth.queries(Q, HQ=8 * G, seed=11, dtype=torch.float16)
    qsl = torch.tensor([0, Q], dtype=torch.int32)
    cache = llama3_cache(512)
    dev = "cuda"
    dec_map = torch.full((pg["num_blocks"],), -1, dtype=torch.int32)
    dec_map[pg["block_table"][0, 0]] = 0
    out = kernels.prefill_paged(st["lay"], q.to(dev), pg["page"].to(dev), 16,
                                pg["block_table"].to(dev), pg["seq_lens"].to(dev), qsl.to(dev), Q, n,
                                dec_map.to(dev), dec_pool_of([st["decoder"]], dev), cache.to(dev),
                                scale)
    lay = st["lay"]
    ks, vs = attend.gather_request(lay, pg["page"], pg["block_table"][0], n, 16)
    cos, sin = rope.cos_sin_from_cache(cache, torch.arange(n), 128)
    s = attend.raw_scores_multi(lay, ks, st["decoder"], q.permute(1, 0, 2), cos, sin, scale,
                                p0=n - Q, dtype=torch.float64)
    p = torch.softmax(s, -1)
    V = attend.dense_v_from_slots(lay, vs, torch.float64).repeat_interleave(G, 0)
    e = (out.cpu().double().permute(1, 0, 2) - p @ V).abs()
    # each weight times its row's ruler is rounded to fp16 once, and so is the output: 2^-11 of
    # sum p |v| each; 1e-4 for the 32-bit scores (|s| < 15)
    assert (e <= 2.0 ** -10 * (p @ V.abs()) + 1e-4).all(), e.max()


def test_four_heads_with_a_workspace_too_small_for_tiles():
    """Four query heads per KV head and a workspace that holds no expanded tiles: the fused kernel,
    whose keys are not split here."""
    st = fitted_store("safe", 200, seed=51)
    pg = paged([st], 16, 4)
    q = synth.queries(40, HQ=32, seed=10, dtype=torch.float16)
    qsl = torch.tensor([0, 40], dtype=torch.int32)
    cache = llama3_cache(512)
    dev = "cuda"
    dec_map = torch.full((pg["num_blocks"],), -1, dtype=torch.int32)
    dec_map[pg["block_table"][0, 0]] = 0
    out = torch.full((40, 32, 128), float("nan"), dtype=torch.float16, device=dev)
    err = torch.zeros(1, dtype=torch.int32, device=dev)
    kernels.prefill_paged(st["lay"], q.to(dev), pg["page"].to(dev), 16,
                          pg["block_table"].to(dev), pg["seq_lens"].to(dev), qsl.to(dev), 40, 200,
                          dec_map.to(dev), dec_pool_of([st["decoder"]], dev), cache.to(dev), SCALE,
                          out=out, error_word=err,
                          workspace=torch.zeros(256, dtype=torch.uint8, device=dev))
    torch.cuda.synchronize()
    want = attend.paged_continuation(st["lay"], pg["page"], pg["block_table"], pg["seq_lens"], qsl,
                                     q.float(), [st["decoder"]], cache, 16, SCALE,
                                     dtype=torch.float64)[0]
    e = (out.float().cpu().double() - want).abs()
    assert int(err.item()) == 0 and e.max() <= 2e-3 and e.mean() <= 1e-3
