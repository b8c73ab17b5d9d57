"""K1 on batches whose tiles are laid end to end and cut into equal ranges (many requests of
different lengths, see the work plan in csrc/ttkv_decode.hip): a workgroup walks the tail of one
request, whole ones and the head of another. Against the CPU oracle, request by request."""
import pytest
import torch

from helpers import dec_pool_of, device_store, fitted_store, llama3_cache, paged
from oracle import attend
from vllm_ttkv import kernels, synth

pytestmark = pytest.mark.gpu
MAX_ABS, MEAN_ABS = 2e-3, 1e-3
SCALE = 128 ** -0.5


def _takes_ranges(lens, H, block_size=16):
    """Whether the device's plan cuts this batch into ranges (the rule of the kernel's work plan)."""
    def up(a, b):
        return -(-a // b)
    target = 2 * torch.cuda.get_device_properties(0).multi_processor_count
    tiles = [max(1, up(n, 64)) for n in lens]
    cap = max(min(258 * block_size // 64, 64), 1)

    def items(m):
        return H * sum(max(1, up(up(n, 64), m)) for n in lens)
    rounds = max(1, up(len(lens) * H, target))
    m = next((m for m in range(1, cap) if items(m) <= rounds * target), cap)
    teams = max(1, target // H)
    units = sum(tiles) + len(lens)
    share = up(units, teams)
    longest = max(min(t, m) for t in tiles)
    return (len(lens) > 1 and units > 2 * teams and share < cap
            and 16 * up(items(m), target) * (longest + 1) > 18 * (share + 1))


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
    assert _takes_ranges(lens, H)
    _batch(cfg, lens, H, G, r1, seed=5, dtype=dtype)


def test_empty_and_undecodable_requests_in_ranges():
    """Empty contexts give zeros and requests without a decoder NaN (error bit 1), at the head of
    a range, in its middle and in a row; the others are unaffected."""
    lens = RAGGED * 9
    assert _takes_ranges(lens, 8)
    got = _batch("safe", lens, 8, 3, 110, seed=6, dtype=torch.float16,
                 empty=(0, 1, 2, 20, 33, 34, 71), lost=(3, 8, 21, 40, 41, 63))
    assert got.shape[0] == 72


def test_one_workspace_for_ranges_and_chunks():
    """A range batch, a uniform one and the range batch again on one workspace: the counters come
    back to zero and the repeat is bit-identical."""
    lens = RAGGED * 9
    assert _takes_ranges(lens, 8) and not _takes_ranges([900] * 5, 8)
    lay = fitted_store("safe", 64, seed=5 + 64)["lay"]
    need = kernels.decode_workspace(lay, 24, len(lens), max(lens), "cuda").numel()
    ws = torch.zeros(need, dtype=torch.uint8, device="cuda")
    a = _batch("safe", lens, 8, 3, 110, seed=7, dtype=torch.float16, workspace=ws)
    _batch("safe", [900] * 5, 8, 3, 110, seed=7, dtype=torch.float16, workspace=ws)
    b = _batch("safe", lens, 8, 3, 110, seed=7, dtype=torch.float16, workspace=ws)
    assert torch.equal(a, b)
    assert int(ws[:65536].abs().sum()) == 0


@pytest.mark.parametrize("cfg,block_size,where,dtype", [
    ("safe", 16, 63, torch.float16), ("safe", 32, 0, torch.bfloat16),
    ("campaign4x", 64, 31, torch.float16), ("safe_fp16", 16, 40, torch.float16),
    ("campaign4x_int4g32", 32, 5, torch.bfloat16)])
def test_a_long_request_among_short_ones(cfg, block_size, where, dtype):
    """One request in more partials than a thread's registers combine: the workgroup that combines
    them weighs them in the tile buffers, and opens its next segment there."""
    print(f"[k1 ranges] {cfg} block {block_size} long at {where} {dtype}", flush=True)
    lens = [70 + 3 * i for i in range(63)]
    lens.insert(where, 14000)
    assert _takes_ranges(lens, 8, block_size)
    st = device_store(cfg, lens, seed=8, block_size=block_size)
    q = synth.queries(64, HQ=24, seed=12, dtype=dtype)
    cache = llama3_cache(16384)
    dev = "cuda"
    out = torch.full((64, 24, 128), float("nan"), dtype=dtype, device=dev)
    err = torch.zeros(1, dtype=torch.int32, device=dev)
    args = (st["play"], q.to(dev), st["page"], block_size, st["block_table"], st["seq_lens"],
            torch.arange(65, dtype=torch.int32, device=dev), 14000, st["dec_map"],
            st["dec_pool"], cache.to(dev), SCALE)
    ws = kernels.decode_workspace(st["play"], 24, 64, 14000, dev, block_size)
    kernels.decode_paged(*args, out=out, error_word=err, workspace=ws)
    got = out.float().cpu()
    kernels.decode_paged(*args, out=out.fill_(0), error_word=err, workspace=ws)
    assert torch.equal(out.float().cpu(), got) and int(err.item()) == 0
    page, bt = st["page"].cpu(), st["block_table"].cpu()
    tol = 1.0 if dtype == torch.float16 else 8.0
    for r in range(64):
        want = attend.paged_decode(st["lay"], page, bt[r:r + 1], torch.tensor([lens[r]]),
                                   torch.arange(2), q[r:r + 1].float(), [st["decoders"][r]],
                                   cache, block_size, SCALE, dtype=torch.float64)
        e = (got[r].double() - want[0]).abs()
        assert e.max() <= tol * MAX_ABS and e.mean() <= tol * MEAN_ABS, (r, lens[r], e.max())
