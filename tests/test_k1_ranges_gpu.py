"""K1 on batches whose tiles are laid end to end and cut into equal ranges (many requests of
different lengths, see the work plan in csrc/ttkv_decode.hip): a workgroup walks the tail of one
request, whole ones and the head of another. Against the CPU oracle, request by request."""
import pytest
import torch

from helpers import dec_pool_of, fitted_store, llama3_cache, paged
from oracle import attend
from vllm_ttkv import kernels, synth

pytestmark = pytest.mark.gpu
MAX_ABS, MEAN_ABS = 2e-3, 1e-3
SCALE = 128 ** -0.5


def _batch(cfg, lens, H, G, r1, seed, dtype, empty=(), lost=(), block_size=16, workspace=None):
    base = {n: fitted_store(cfg, n, seed=seed + n, r1=r1, H_=H) for n in sorted(set(lens))}
    stores = [base[n] for n in lens]
    B = len(lens)
    pg = paged(stores, block_size, seed)
    q = synth.queries(B, HQ=H * G, seed=seed, dtype=dtype)
    dec_map = torch.full((pg["num_blocks"],), -1, dtype=torch.int32)
    for r in range(B):
        if r not in lost:
            dec_map[pg["block_table"][r, 0]] = r
    seq = pg["seq_lens"].clone()
    seq[list(empty)] = 0
    dev = "cuda"
    cache = llama3_cache(2048)
    out = torch.full((B, H * G, 128), float("nan"), dtype=dtype, device=dev)
    err = torch.zeros(1, dtype=torch.int32, device=dev)
    kernels.decode_paged(stores[0]["lay"], q.to(dev), pg["page"].to(dev), block_size,
                         pg["block_table"].to(dev), seq.to(dev),
                         torch.arange(B + 1, dtype=torch.int32, device=dev), max(lens),
                         dec_map.to(dev), dec_pool_of([s["decoder"] for s in stores], dev),
                         cache.to(dev), SCALE, out=out, error_word=err, workspace=workspace)
    torch.cuda.synchronize()
    assert int(err.item()) == (1 if lost else 0)
    got = out.float().cpu()
    tol = 1.0 if dtype == torch.float16 else 8.0     # bf16 rounds the output 8 times coarser
    for r in range(B):
        if r in empty:
            assert not got[r].any(), r
        elif r in lost:
            assert torch.isnan(got[r]).all(), r
        else:
            want = attend.paged_decode(stores[0]["lay"], pg["page"], pg["block_table"][r:r + 1],
                                       seq[r:r + 1], torch.arange(2), q[r:r + 1].float(),
                                       [stores[r]["decoder"]], cache, block_size, SCALE,
                                       dtype=torch.float64)
            e = (got[r].double() - want[0]).abs()
            assert e.max() <= tol * MAX_ABS and e.mean() <= tol * MEAN_ABS, (r, lens[r], e.max())
    return got


RAGGED = [1500, 1, 17, 64, 65, 130, 257, 900]


@pytest.mark.parametrize("cfg,H,G,r1,dtype", [
    ("safe", 8, 3, 110, torch.float16), ("campaign4x", 8, 3, 110, torch.bfloat16),
    ("safe", 8, 4, 96, torch.bfloat16), ("tight", 8, 1, 64, torch.float16),
    ("safe", 4, 8, 126, torch.float16), ("safe", 3, 2, 110, torch.float16)])
def test_ragged_requests_in_ranges(cfg, H, G, r1, dtype):
    print(f"[k1 ranges] {cfg} H={H} G={G} r1={r1} {dtype}", flush=True)
    lens = RAGGED * (8 if H == 8 else 20)
    _batch(cfg, lens, H, G, r1, seed=5, dtype=dtype)


def test_empty_and_undecodable_requests_in_ranges():
    """Empty contexts give zeros and requests without a decoder NaN (error bit 1), at the head of
    a range, in its middle and in a row; the others are unaffected."""
    lens = RAGGED * 9
    got = _batch("safe", lens, 8, 3, 110, seed=6, dtype=torch.float16,
                 empty=(0, 1, 2, 20, 33, 34, 71), lost=(3, 8, 21, 40, 41, 63))
    assert got.shape[0] == 72


def test_one_workspace_for_ranges_and_chunks():
    """A range batch, a uniform one and the range batch again on one workspace: the counters come
    back to zero and the repeat is bit-identical."""
    lens = RAGGED * 9
    lay = fitted_store("safe", 64, seed=5 + 64)["lay"]
    need = kernels.decode_workspace(lay, 24, len(lens), max(lens), "cuda").numel()
    ws = torch.zeros(need, dtype=torch.uint8, device="cuda")
    a = _batch("safe", lens, 8, 3, 110, seed=7, dtype=torch.float16, workspace=ws)
    _batch("safe", [900] * 5, 8, 3, 110, seed=7, dtype=torch.float16, workspace=ws)
    b = _batch("safe", lens, 8, 3, 110, seed=7, dtype=torch.float16, workspace=ws)
    assert torch.equal(a, b)
    assert int(ws[:65536].abs().sum()) == 0
