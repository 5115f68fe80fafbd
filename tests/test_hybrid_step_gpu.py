"""One token per row in one launch (mui_hybrid_step) against the float64 oracle and, for what it leaves in the caches, against
the launches it stands for."""
import pytest
import torch

from muillm_amd import _lib, hybrid_ops as ops
from oracle import zufadra as oracle

pytestmark = pytest.mark.gpu
DEV = "cuda"
REL = {torch.bfloat16: 2e-2, torch.float16: 3e-3}  # of the largest value: 16-bit queries, keys, probabilities and outputs (as for the separate launches)

CASES = [  # heads, kv_heads, dim, vdim, rot, window, keep_first, softcap, scale, gated, gains
    (6, 2, 40, 24, 16, 37, 3, 7.5, 0.2, True, True), (4, 4, 64, 64, 64, 0, 0, 0.0, 0.12, False, True), (32, 8, 128, 128, 64, 4096, 64, 30.0, 0.09, True, True),
    (8, 2, 96, 128, 0, 130, 70, 20.0, 0.1, True, False), (18, 1, 32, 40, 32, 65, 1, 11.0, 0.2, True, True), (2, 1, 200, 256, 40, 64, 64, 0.0, 0.07, True, True),
    (3, 3, 8, 8, 8, 1, 0, 2.0, 0.4, False, False), (40, 2, 72, 16, 24, 0, 0, 5.0, 0.15, True, True)]


def _inputs(dtype, case, seed, batch, capacity):
    heads, kv_heads, dim, vdim, rot = CASES[case][:5]
    g = torch.Generator().manual_seed(seed)
    rand = lambda *s: torch.randn(*s, generator=g)
    widths = (heads * dim, kv_heads * dim, kv_heads * vdim, heads * vdim)
    proj = (1.5 * rand(batch, 1, sum(widths))).to(dtype)
    gains = [(1 + 0.3 * rand(w)).to(dtype) for w in widths[:2]] if CASES[case][10] else [None, None]
    k, v = (rand(batch, capacity, w).to(dtype) for w in widths[1:3])
    freq = oracle.frequencies(rot, 50.0) if rot else torch.zeros(0, dtype=torch.float64)
    return proj, gains, k, v, freq, widths


def _step(case, proj, gains, k, v, freq, slot, pads):
    heads, kv_heads, dim, vdim, rot, window, keep, softcap, scale, gated, _ = CASES[case]
    dev = lambda x: None if x is None else x.to(DEV)
    return ops.hybrid_step(dev(proj), heads, kv_heads, dim, vdim, *map(dev, gains), 0.2, dev(freq), torch.tensor([slot], device=DEV), dev(pads),
                           k, v, gated, scale, softcap, window, keep)


def _reference(case, proj, gains, k, v, freq, slot, pads, widths):
    heads, kv_heads, dim, vdim, rot, window, keep, softcap, scale, gated, _ = CASES[case]
    out = []
    for b in range(proj.shape[0]):
        first = int(pads[b])
        q, nk, nv, gate = proj[b, 0].double().split(widths)
        if gains[0] is not None:
            q, nk = oracle.rms(q[None], 0.2)[0] * gains[0].double(), oracle.rms(nk[None], 0.2)[0] * gains[1].double()
        pos = torch.tensor([max(slot - first, 0)])
        q, nk = (oracle.rotate_pairs(x.reshape(1, -1, dim), pos, freq) for x in (q, nk))
        keys = torch.cat([k[b, first:slot].double().reshape(-1, kv_heads, dim), nk])
        values = torch.cat([v[b, first:slot].double().reshape(-1, kv_heads, vdim), nv.reshape(1, kv_heads, vdim)])
        y = oracle.attention(q, keys, values, scale, softcap, window, keep, slot - first).reshape(-1)
        out.append(y * torch.sigmoid(gate) if gated else y)
    return torch.stack(out)


@pytest.mark.parametrize("dtype", list(REL))
@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("capacity", [1, 64, 65, 128, 130, 192, 256])
def test_step(dtype, case, capacity):
    heads, kv_heads, dim, vdim, rot, window, keep = CASES[case][:7]
    if not _lib.load().mui_hybrid_step_serves(ops.dtype_code(dtype), 3, heads, kv_heads, dim, vdim, window, keep, capacity):
        assert capacity > 128 and max(dim, vdim) > 128
        return
    for slot in sorted({0, capacity // 2, max(capacity - 64, 0), capacity - 1}):
        pads = torch.tensor([0, slot // 3, slot])
        proj, gains, k, v, freq, widths = _inputs(dtype, case, 7 * slot + capacity, 3, capacity)
        k[:, slot:], v[:, slot:] = float("nan"), float("nan")  # what the caches hold from the slot on is never used
        kc, vc, kd, vd = (x.to(DEV) for x in (k, v, k.clone(), v.clone()))
        got = _step(case, proj, gains, kc, vc, freq, slot, pads)
        ref = _reference(case, proj, gains, k, v, freq, slot, pads, widths)
        assert bool(torch.isfinite(got).all())
        err = float((got[:, 0].cpu().double() - ref).abs().max() / ref.abs().max())
        assert err <= REL[dtype], (slot, err)
        dev = lambda x: None if x is None else x.to(DEV)
        ops.hybrid_prepare(dev(proj), heads, kv_heads, dim, vdim, *map(dev, gains), 0.2, dev(freq), torch.tensor([slot], device=DEV), dev(pads), kd, vd)
        assert torch.equal(vc.view(torch.int16), vd.view(torch.int16))
        rest = torch.arange(capacity) != slot
        assert torch.equal(kc[:, rest].view(torch.int16), kd[:, rest].view(torch.int16))
        # the new key: sums of squares in another order, so a unit in the last place at most
        assert torch.allclose(kc[:, slot].float(), kd[:, slot].float(), rtol=2 ** -7 if dtype == torch.bfloat16 else 2 ** -10, atol=1e-6)


@pytest.mark.parametrize("dtype", list(REL))
@pytest.mark.parametrize("slot,pads", [(100, (0, 101)), (128, (0, 3)), (300, (0, 3)), (-1, (0, 0)), (99, (99, 200))])
def test_slots_outside_the_cache_and_rows_that_have_not_begun(dtype, slot, pads):
    """As the separate launches: nothing is stored outside, a row without a visible key gives zeros."""
    case, capacity = 0, 128
    heads, kv_heads, dim, vdim, rot, window, keep, softcap, scale, gated, _ = CASES[case]
    proj, gains, k, v, freq, widths = _inputs(dtype, case, slot + 9, 2, capacity)
    pads = torch.tensor(pads)
    kc, vc, kd, vd = (x.to(DEV) for x in (k, v, k.clone(), v.clone()))
    got = _step(case, proj, gains, kc, vc, freq, slot, pads)
    at, dev = torch.tensor([slot], device=DEV), lambda x: x.to(DEV)
    q = ops.hybrid_prepare(dev(proj), heads, kv_heads, dim, vdim, *map(dev, gains), 0.2, dev(freq), at, dev(pads), kd, vd)
    want = ops.hybrid_attention(q, kd, vd, dev(proj)[..., sum(widths[:3]):], at, dev(pads), heads, kv_heads, scale, softcap, window, keep)
    assert float((got.float() - want.float()).abs().max()) <= REL[dtype] * max(float(want.float().abs().max()), 1e-3)
    assert torch.equal(vc, vd) and torch.allclose(kc.float(), kd.float(), rtol=2 ** -7, atol=1e-6)


def test_what_is_left_to_the_separate_launches():
    bf16 = _lib.MUI_DTYPE_BF16
    serves = lambda dtype, *a, batch=2: _lib.load().mui_hybrid_step_serves(dtype, batch, *a)
    assert serves(bf16, 32, 8, 128, 128, 4096, 64, 256) and not serves(bf16, 32, 8, 128, 128, 4096, 64, 257)
    assert serves(bf16, 32, 8, 128, 128, 192, 64, 1 << 20) and not serves(bf16, 32, 8, 128, 128, 193, 64, 1 << 20)
    assert not serves(_lib.MUI_DTYPE_F32, 4, 4, 64, 64, 0, 0, 64) and not serves(bf16, 4, 4, 20, 12, 9, 2, 64) and not serves(bf16, 2, 2, 16, 264, 2, 1, 64)
    assert serves(bf16, 32, 8, 128, 128, 0, 0, 256, batch=32) and not serves(bf16, 32, 8, 128, 128, 0, 0, 256, batch=64) and serves(bf16, 32, 8, 128, 128, 0, 0, 128, batch=64)
    assert serves(bf16, 4, 4, 256, 64, 0, 0, 128) and not serves(bf16, 4, 4, 256, 64, 0, 0, 129)
    assert not serves(bf16, 5, 2, 64, 64, 0, 0, 64) and not serves(bf16, 4, 4, 64, 64, -1, 0, 64) and not serves(bf16, 4, 4, 64, 64, 0, 0, 64, batch=0) and not serves(bf16, 4, 4, 64, 64, 2**31 - 1, 2**31 - 1, 4096)
    proj, gains, k, v, freq, _ = _inputs(torch.bfloat16, 1, 0, 2, 64)
    k, v = k.to(DEV), v.to(DEV)
    assert _step(1, proj.repeat(1, 2, 1), gains, k, v, freq, 3, None) is None  # two tokens per row
    off = torch.zeros(k.numel() + 1, dtype=k.dtype, device=DEV)[1:].view(k.shape)
    assert _step(1, proj, gains, off, v, freq, 3, None) is None  # a cache off the 16-byte grid
    assert _step(1, proj, gains, k, v, freq, 3, None) is not None
