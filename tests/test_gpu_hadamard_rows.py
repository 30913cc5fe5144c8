"""OnlineHadamard + Quantizer of a few hundred rows at most, of 64 or 128 values behind a table: one workgroup per row, one wave per 16
rows of the table.  Codes and scales must carry the bits that the same rows get inside a batch of more rows than two per CU, which
four waves a row transform."""
import pytest
import torch

import quarot_amd

pytestmark = pytest.mark.gpu
MANY = 1100                                                 # more than two rows on each of 256 CUs, by a margin


def _bits(p):
    return p.quantized_x, p.scales_x.view(torch.int16)


# 64 x 172 / 156 / 140 / 108 (last tile of 16 rows half empty), 128 x 108 / 60 / 52 / 40 / 36
@pytest.mark.parametrize("n", [11008, 9984, 8960, 6912, 13824, 7680, 6656, 5120, 4608])
@pytest.mark.parametrize("signs", [True, False])           # the reference's table, and one whose entries are not +-1
def test_few_rows_have_the_bits_of_many(n, signs):
    gen = torch.Generator(device="cuda").manual_seed(n)
    table, K = quarot_amd.functional.hadamard.get_hadK(n)
    hadK = table.to("cuda").half()
    if not signs:
        hadK = (hadK * (torch.rand(K, K, generator=gen, device="cuda") + 0.5)).half()
    x = torch.randn(MANY, n, device="cuda", generator=gen)
    x[:, torch.randperm(n, generator=gen, device="cuda")[:n // 100]] *= 20
    x[0], x[1, 3], x[2, n - 1] = 0, float("inf"), float("nan")
    x[3], x[4], x[5] = x[3] * 1e-6, (x[4] * 20000).clamp(-60000, 60000), -float("inf")
    x = x.half()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert MANY > 2 * cus
    for clip in (1.0, 0.83):
        many = _bits(quarot_amd.hadamard_quantize(x, hadK, K, clip_ratio=clip))
        for rows in (1, 2, 7, 48, cus, cus + 1, 2 * cus, 2 * cus + 1):
            few = _bits(quarot_amd.hadamard_quantize(x[:rows].contiguous(), hadK, K, clip_ratio=clip))
            assert torch.equal(few[0], many[0][:rows]) and torch.equal(few[1].view(-1), many[1][:rows].view(-1)), (rows, clip)
        end = _bits(quarot_amd.hadamard_quantize(x[MANY - 33:].contiguous(), hadK, K, clip_ratio=clip))
        assert torch.equal(end[0], many[0][-33:]) and torch.equal(end[1].view(-1), many[1][-33:].view(-1))
