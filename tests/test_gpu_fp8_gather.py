"""The fp8 gather (nia_dequant_gather_fp8, and the rows nia_prefill_paged_fp8 attends) bit for
bit against code * scale rounded to bf16: block sizes that leave partial pieces of a
workgroup, contexts inside a block, invalid blocks (zero rows), rows past a context left
alone, and caches off a 16-byte boundary."""
import pytest
import torch

from nano_inference_amd import _lib

pytestmark = pytest.mark.gpu


def _shifted(t, shift):
    """t on the GPU with its first byte ``shift`` bytes past a 256-byte boundary."""
    buf = torch.zeros(t.numel() + 256, dtype=torch.uint8, device="cuda")
    out = buf[shift:shift + t.numel()].view(t.shape)
    out.copy_(t)
    return out


@pytest.mark.parametrize("shift", [0, 2])
@pytest.mark.parametrize("bs,hkv,lens", [(1, 3, [1, 7]), (5, 1, [4, 5, 26]), (16, 8, [0, 513, 40]),
                                         (100, 3, [99, 301]), (256, 4, [257, 1])])
def test_gather(bs, hkv, lens, shift):
    print(f"fp8 gather bs={bs} hkv={hkv} lens={lens} shift={shift}", flush=True)
    d, n, mb = 128, len(lens), max(-(-x // bs) for x in lens) + 1
    nb = n * mb
    g = torch.Generator().manual_seed(bs + shift)
    codes = [torch.randint(0, 256, (nb, hkv, bs, d), generator=g).to(torch.uint8) for _ in range(2)]
    for c in codes:
        c[(c & 0x7F) == 0x7F] = 0x3A  # no NaN codes
    scales = [torch.rand((nb, hkv, bs), generator=g) + 0.01 for _ in range(2)]
    tables = torch.randperm(nb, generator=g).view(n, mb).to(torch.int32)
    tables[0, 0] = -1
    stride = mb * bs + 3
    gpu = [_shifted(c, shift) for c in codes] + [s.cuda() for s in scales]
    out = [torch.full((n * stride, hkv, d), 7.0, dtype=torch.bfloat16, device="cuda")
           for _ in range(2)]
    ctx = torch.tensor(lens, dtype=torch.int64, device="cuda")
    tb = tables.cuda()
    st = _lib.load().nia_dequant_gather_fp8(
        *(t.data_ptr() for t in gpu), tb.data_ptr(), mb, mb, ctx.data_ptr(), n, hkv, d, bs, nb,
        out[0].data_ptr(), out[1].data_ptr(), stride, torch.cuda.current_stream().cuda_stream)
    assert st == _lib.OK
    for o, c, s in zip(out, codes, scales):
        rows = (c.view(torch.float8_e4m3fn).float() * s.unsqueeze(-1)).to(torch.bfloat16)
        exp = torch.full((n, stride, hkv, d), 7.0, dtype=torch.bfloat16)
        for i, length in enumerate(lens):
            for t in range(length):
                b = int(tables[i, t // bs])
                exp[i, t] = 0.0 if b < 0 else rows[b, :, t % bs]
        assert torch.equal(o.cpu().view(torch.int16),
                           exp.view(n * stride, hkv, d).view(torch.int16))


def test_wide_table_of_single_rows():
    """More table entries than one grid dimension has workgroups of 256 threads (2^24): a key a
    block and one KV head."""
    d, mb, length = 128, (1 << 24) + 3, 7
    g = torch.Generator().manual_seed(9)
    codes = torch.randint(0, 120, (8, 1, 1, d), generator=g).to(torch.uint8)
    scale = torch.rand((8, 1, 1), generator=g) + 0.01
    table = torch.zeros(mb, dtype=torch.int32)
    table[:length] = torch.randperm(8, generator=g)[:length]
    tb, cg, sg = table.cuda(), codes.cuda(), scale.cuda()
    out = [torch.full((length, 1, d), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    ctx = torch.tensor([length], dtype=torch.int64, device="cuda")  # no row past it is written
    st = _lib.load().nia_dequant_gather_fp8(
        cg.data_ptr(), cg.data_ptr(), sg.data_ptr(), sg.data_ptr(), tb.data_ptr(), mb, mb,
        ctx.data_ptr(), 1, 1, d, 1, 8, out[0].data_ptr(), out[1].data_ptr(), mb,
        torch.cuda.current_stream().cuda_stream)
    assert st == _lib.OK
    rows = (codes.view(torch.float8_e4m3fn).float() * scale.unsqueeze(-1)).to(torch.bfloat16)
    exp = rows[table[:length].long(), 0]
    assert all(torch.equal(o.cpu(), exp) for o in out)
