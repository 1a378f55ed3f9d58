"""The fused QK step at the edges of its row layouts: a wave a row and groups of eight, on both
sides of their bound, rows that do not fill a group, a token's rows in one wave or spread over
several, query and key rows in one group, and views whose rows are not 16-byte aligned
(element accesses).  Bars as in
test_gpu_qk_rope; cache rows bit-identical to the write of the kernel's own k and the
input v."""
import pytest
import torch

from nano_inference_amd import ops
from oracle import fp8_kv
from oracle import qk_rope as O
from oracle import reference_attention as ref

from tests.test_gpu_qk_rope import D, EPS, _compare

pytestmark = pytest.mark.gpu


def _rows(x, shift):
    """x (n, heads, D) on the GPU, its first element ``shift`` elements into a buffer whose
    token stride is a multiple of 16 bytes only for shift 0."""
    n, h, _ = x.shape
    buf = torch.zeros(n * (h * D + shift) + shift, dtype=x.dtype, device="cuda")
    out = buf[shift:].as_strided((n, h, D), (h * D + shift, D, 1), shift)
    out.copy_(x)
    return out


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("store", ["bf16", "fp8", "f32"])
@pytest.mark.parametrize("n,h,hkv,mrope", [(1, 16, 8, False), (3, 7, 1, False), (33, 28, 4, True),
                                           (700, 32, 8, False), (2051, 3, 1, False),
                                           # a wave a row up to 5120 rows, groups past them
                                           (128, 32, 8, True), (129, 32, 8, False),
                                           (161, 31, 1, False), (2561, 1, 1, False)])
def test_row_groups(n, h, hkv, mrope, store, shift):
    print(f"rope rows n={n} h={h} hkv={hkv} mrope={mrope} {store} shift={shift}", flush=True)
    dtype = torch.float32 if store == "f32" else torch.bfloat16
    g = torch.Generator().manual_seed(n + h + shift)
    q, k, v = (torch.randn(n, m, D, generator=g).to(dtype) for m in (h, hkv, hkv))
    qw, kw = ((torch.randn(D, generator=g) * 0.3 + 1).to(dtype) for _ in range(2))
    pos = torch.randint(0, 40000, (3, 1, n) if mrope else (1, n), generator=g)
    sec = (16, 24, 24) if mrope else None
    bs, nb = 16, -(-n // 16) + 2
    slots = torch.randperm(nb * bs, generator=g)[:n]
    slots[n // 2] = -1 if n > 1 else slots[0]
    freqs = O.inv_freq(D, 1e6)
    eq, ek = O.qk_norm_rope(q[None], k[None], qw, kw, EPS, pos, freqs, sec)
    qg, kg, vg = (_rows(t, shift) for t in (q, k, v))
    ct = torch.uint8 if store == "fp8" else dtype
    kc, vc = (torch.zeros(nb, hkv, bs, D, dtype=ct) for _ in range(2))
    ks, vs = (torch.zeros(nb, hkv, bs) for _ in range(2))
    gpu = [t.cuda() for t in (kc, vc, slots, ks, vs)]
    ops.qk_norm_rope_kv_write(qg, kg, vg, qw.cuda(), kw.cuda(), EPS,
                              pos.view(3, n).cuda() if mrope else pos.view(n).cuda(),
                              freqs.cuda(), sec, *gpu[:3], *(gpu[3:] if store == "fp8" else ()))
    _compare(qg[None], eq, "q")
    _compare(kg[None], ek, "k")
    assert torch.equal(vg.cpu(), v), "v must not change"
    k_out = kg.cpu().contiguous()
    if store == "fp8":
        fp8_kv.kv_write_loop_fp8(k_out[None], v[None], kc, vc, ks, vs, slots[None])
        assert torch.equal(gpu[3].cpu(), ks) and torch.equal(gpu[4].cpu(), vs), "scales"
    else:
        ref.kv_write_loop(k_out[None], v[None], kc, vc, slots[None])
    bits = torch.uint8 if store == "fp8" else (torch.int32 if store == "f32" else torch.int16)
    assert torch.equal(gpu[0].cpu().view(bits), kc.view(bits)), "k cache bits"
    assert torch.equal(gpu[1].cpu().view(bits), vc.view(bits)), "v cache bits"
