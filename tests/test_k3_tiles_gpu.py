"""K3 over many tokens (tiles of up to 16 tokens of one request, from 208 tokens on and 3 more for
every further request) on the GPU: at the edges of tiles and requests, the float stages within the rounding of their own sums against 64 bits, and every byte exactly the
oracle's from the kernel's own projection and residual."""
import pytest
import torch

from helpers import D, dec_pool_of
from oracle import codec, coef_modes, encode
from oracle.layout import layout_for_config
from vllm_ttkv import kernels
from vllm_ttkv.layout import config_named

pytestmark = pytest.mark.gpu
DEV = "cuda"
EPS = 2.0 ** -24


def _decoder(r1, H, seed):
    """A codec-form decoder (int8 rows times fp16 rulers) with every rank active."""
    g = torch.Generator().manual_seed(seed)
    q = torch.randint(-127, 128, (r1, H * D), generator=g).float()
    q[:, 0] = 127.0                       # as in every codec row, the largest |q| is 127
    return q * (torch.rand(r1, generator=g) * 0.02 + 0.005).half().float()[:, None]


def _tiled(counts):
    return sum(counts) >= 208 + 3 * (len(counts) - 1)


def _case(cfg, r1, H, counts, dtype, seed, fit=False):
    lay = layout_for_config(config_named(cfg), r1=r1, H=H)
    g = torch.Generator().manual_seed(seed)
    N, B = sum(counts), len(counts)
    decs = [_decoder(r1, H, seed + r) for r in range(B)]
    pinvs = [encode.pinv(d) for d in decs]
    K = torch.cat([torch.randn(m, r1, generator=g) @ d + 0.2 * torch.randn(m, H * D, generator=g)
                   for m, d in zip(counts, decs)]).to(dtype)
    V = torch.randn(N, H * D, generator=g).to(dtype)
    req = torch.cat([torch.full((m,), r) for r, m in enumerate(counts)])
    slots = torch.randperm(N + 40, generator=g)[:N]
    qsl = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)), dtype=torch.int32)
    kw = {}
    if fit:
        kw = dict(coeff_q_in=torch.randint(-127, 128, (N, r1), generator=g).to(torch.int8).to(DEV),
                  coeff_scale_in=(torch.rand(N, generator=g) * 0.02 + 1e-3).to(DEV))
    return dict(lay=lay, K=K, V=V, decs=decs, pinvs=pinvs, req=req, slots=slots, qsl=qsl, kw=kw,
                H=H)


def _run(c, slots=None, dec_map=None, used=None, views=None, n_slots=None):
    lay, N, B, H = c["lay"], len(c["req"]), len(c["decs"]), c["H"]
    page = torch.zeros(n_slots or N + 40, lay.compressed_bytes_per_token(), dtype=torch.uint8,
                       device=DEV)
    bt = torch.arange(B, dtype=torch.int32, device=DEV).reshape(B, 1)
    if dec_map is None:
        dec_map = torch.arange(B, dtype=torch.int32)
    c_out = torch.zeros(N, lay.r1, device=DEV)
    r_out = torch.zeros(N, H * D, device=DEV)
    err = torch.zeros(1, dtype=torch.int32, device=DEV)
    v = views or {n: c[n].reshape(N, H, D).to(DEV) for n in "KV"}
    kernels.write_paged(lay, v["K"], v["V"],
                        (c["slots"] if slots is None else slots).to(DEV), c["qsl"].to(DEV), bt,
                        dec_map.to(DEV), dec_pool_of(c["decs"], DEV),
                        torch.stack([p.t() for p in c["pinvs"]]).contiguous().to(DEV), page,
                        coeff_out=c_out, resid_out=r_out, error_word=err, dec_used=used, **c["kw"])
    torch.cuda.synchronize()
    return page.cpu(), c_out.cpu(), r_out.cpu(), int(err.item())


def _want(c, coef, R):
    """The blobs [N, C] the oracle packs from the kernel's own c and R, and R in 64 bits."""
    lay, N, H = c["lay"], len(c["req"]), c["H"]
    if c["kw"]:
        q, s32 = c["kw"]["coeff_q_in"].cpu(), c["kw"]["coeff_scale_in"].cpu().reshape(-1, 1)
        vals, s = q.float() * s32, s32.half().reshape(-1)
    elif lay.qbits == 8:
        q, s32 = encode.quantise_coeffs(coef)
        vals, s = q.float() * s32.reshape(-1, 1), s32.to(torch.float16).reshape(-1)
    else:
        vals, q, s = coef_modes.quantise(coef, lay.qbits)
    rec = torch.stack([vals[i].double() @ c["decs"][r].double() for i, r in enumerate(c["req"])])
    mag = torch.stack([vals[i].double().abs() @ c["decs"][r].double().abs()
                       for i, r in enumerate(c["req"])])

    def rows(x):
        return x.reshape(N, H, D).permute(1, 0, 2).reshape(H * N, D)
    ks = encode.k_slots_from(lay, q, s, codec.build_rows(rows(R), lay.res_k, lay.res_bits))
    vs = encode.v_slots_from(lay, encode.encode_v(c["V"].float().reshape(N, H, D).permute(1, 0, 2)
                                                  .contiguous(), lay))
    return torch.cat([ks, vs], 1), c["K"].double() - rec, mag


CASES = [
    # (config, r1, KV heads, tokens per request, dtype, from a fit)
    ("safe", 110, 8, [208], torch.float32, False),            # whole tiles
    ("safe", 110, 8, [207], torch.float16, False),            # one token short of tiles
    ("safe", 110, 8, [223], torch.bfloat16, False),           # a 15-token last tile
    ("safe", 110, 8, [192], torch.float32, False),            # token by token
    ("campaign4x", 110, 8, [1, 1, 1, 218], torch.float16, False),  # decodes, then a chunk
    ("campaign4x", 110, 8, [218, 1, 17, 1], torch.float16, False),  # and behind it
    ("tight", 64, 8, [5, 200, 17], torch.float16, False),      # partly filled tiles
    ("tight", 64, 8, [5, 190, 17], torch.float16, False),      # two tokens short of tiles
    ("safe", 7, 2, [1] * 20 + [187, 75, 3], torch.float16, False),  # a small rank
    ("safe", 16, 1, [1] * 70 + [400, 0, 3, 2], torch.float16, False),  # spans past one wave's lanes
    ("safe", 200, 4, [213], torch.float32, False),             # ranks past 128
    ("safe", 96, 3, [209], torch.float16, False),              # H * d / 4 not a multiple of 64
    ("safe", 110, 1, [209], torch.float16, False),
    ("safe_fp16", 110, 8, [197, 20], torch.float16, False),
    ("campaign4x_int4g32", 110, 8, [197, 20], torch.bfloat16, False),
    ("campaign4x_int4g32", 66, 8, [212], torch.float16, False),
    ("safe", 110, 8, [150, 61], torch.float16, True),          # fits' own coefficients
    ("safe", 16, 1, [100, 16600], torch.float16, False),       # two launches of each kernel
]


@pytest.mark.parametrize("cfg,r1,H,counts,dtype,fit", CASES)
def test_tiles(cfg, r1, H, counts, dtype, fit):
    print(f"[k3 tiles] {cfg} r1={r1} H={H} {counts} {dtype} fit={fit}", flush=True)
    c = _case(cfg, r1, H, counts, dtype, seed=r1 + sum(counts), fit=fit)
    page, coef, R, err = _run(c)
    assert err == 0
    K = c["K"].double()
    if not fit:
        want = torch.stack([K[i] @ c["pinvs"][r].double() for i, r in enumerate(c["req"])])
        mag = torch.stack([K[i].abs() @ c["pinvs"][r].double().abs()
                           for i, r in enumerate(c["req"])])
        # no chain of fp32 additions is longer than 16 MFMA steps of 4 products and 4 more
        assert ((coef.double() - want).abs() <= 72 * EPS * mag).all()
    blob, R64, mag = _want(c, coef, R)
    # at most R / 8 MFMA steps of 4 products per accumulator, the c * cs product and the key
    bound = (max(r1 // 2, 32) + 8) * EPS * (mag + K.abs())
    assert ((R.double() - R64).abs() <= bound).all()
    nbad = int((page[c["slots"]] != blob).sum())
    assert nbad == 0, f"{nbad} of {blob.numel()} bytes differ"
    untouched = torch.ones(page.shape[0], dtype=torch.bool)
    untouched[c["slots"]] = False
    assert int(page[untouched].abs().sum()) == 0


def test_skipped_and_refused_tokens_inside_tiles():
    """Inside one tile: padded tokens are skipped silently, a slot past the cache and a request
    without a decoder are refused with their bits, and the others' bytes are the same as without
    them; the use flags name the decoders that were used."""
    counts = [40, 8, 170]
    c = _case("safe", 110, 8, counts, torch.float16, seed=3)
    clean, _, _, err = _run(c)
    assert err == 0
    slots = c["slots"].clone()
    slots[50] = -1
    slots[57:60] = -1
    slots[61] = clean.shape[0]
    used = torch.zeros(3, dtype=torch.int32, device=DEV)
    page, _, _, err = _run(c, slots=slots, dec_map=torch.tensor([0, -1, 2], dtype=torch.int32),
                           used=used)
    assert err == 4 | 1
    keep = torch.ones(sum(counts), dtype=torch.bool)
    keep[40:48] = False
    keep[[50, 57, 58, 59, 61]] = False
    assert torch.equal(page[c["slots"][keep]], clean[c["slots"][keep]])
    assert int(page[c["slots"][~keep]].abs().sum()) == 0
    assert used.tolist() == [1, 0, 1]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_rows_without_alignment(dtype):
    """Keys and values as views of wider rows at an odd offset: the bytes of packed ones."""
    c = _case("safe", 110, 8, [140, 83], dtype, seed=5)
    assert _tiled([140, 83])
    want, coef, R, err = _run(c)
    assert err == 0
    wide = {}
    for name in ("K", "V"):
        x = c[name].to(DEV)
        buf = torch.zeros(x.shape[0], x.shape[1] + 3, dtype=dtype, device=DEV)
        buf[:, 1:1 + x.shape[1]] = x
        wide[name] = buf[:, 1:1 + x.shape[1]].unflatten(1, (8, D))
        assert wide[name].data_ptr() % 16 and wide[name].stride(0) == 8 * D + 3
    page, coef2, R2, err = _run(c, views=wide)
    assert err == 0 and torch.equal(page, want)
    assert torch.equal(coef2, coef) and torch.equal(R2, R)


def test_tokens_outside_every_request():
    """Tokens before the first request and after the last: refused, or skipped where they are
    padding; the requests' own bytes are those of a call without them."""
    c = _case("safe", 110, 8, [100, 125], torch.float16, seed=8)
    want, _, _, err = _run(c)
    assert err == 0 and _tiled([100, 125])
    more = dict(c)
    for name in ("K", "V"):
        x = c[name]
        more[name] = torch.cat([x[:5], x, x[-9:]])
    more["qsl"] = c["qsl"] + 5
    used = c["slots"]
    free = torch.tensor([i for i in range(225 + 40) if i not in set(used.tolist())])
    for outside, bits in ((torch.full((14,), -1), 0), (free[:14], 1)):
        slots = torch.cat([outside[:5], used, outside[5:]])
        page, _, _, err = _run(dict(more, slots=slots, req=torch.zeros(239)), n_slots=265)
        assert err == bits
        assert torch.equal(page, want)
