"""The stand-alone quantize from index lists (asym_quantize_list_kernel) against the column map's path on the same lists: any
order, lists that overlap or leave the row, group counts at the edges of a workgroup's lanes, more rows than workgroups,
rows with NaN, infinities, both zeros, one value only, and ranges beyond the storage type.  Same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _lists(kind, cols, num_fp, g):
    perm = torch.randperm(cols, generator=g)
    fp, ints = perm[:num_fp], perm[num_fp:].sort()[0]
    if kind == "shuffled":
        ints = ints[torch.randperm(len(ints), generator=g)]
    elif kind == "overlapping":
        ints = torch.randint(0, cols, (len(ints),), generator=g)
    elif kind == "outside":
        ints = ints * 2 - cols // 2
        fp = fp - 3
    return ints.to(DEV), fp.to(DEV)


@pytest.mark.parametrize("kind", ["ascending", "shuffled", "overlapping", "outside"])
@pytest.mark.parametrize("rows,cols,num_fp", [(1, 8, 0), (9, 40, 8), (5, 2048, 0), (600, 2056, 256), (33, 4096, 128), (7, 4104, 8),
                                              (1030, 1064, 40), (11, 8192, 0), (3, 8192, 7680), (4, 4096, 4088), (9, 11008, 256),
                                              (3, 16384, 0), (200, 16392, 512), (520, 16392, 512), (2, 32768, 256), (2, 32768, 32760)])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_same_bits_as_the_column_map(kind, rows, cols, num_fp, bits, dtype):
    import quik
    from quik_amd import asymmetric
    g = torch.Generator().manual_seed(rows + cols + num_fp)
    ints, fp = _lists(kind, cols, num_fp, g)
    x = torch.randn(rows, cols, generator=g)
    for r, v in ((0, float("nan")), (1, float("inf")), (2, -float("inf"))):
        x[r % rows, (r * 5 + 1) % cols] = v
    if rows > 8:
        x[4], x[5], x[6] = 0.0, 2.5, x[6].abs()
        x[6, ::3] = -0.0
        x[7] *= 6e4
        x[8] = float("nan")
    x = x.to(dtype).to(DEV)
    got = quik.asymmetric.quantize(x, ints, fp, bits)
    want = asymmetric.quantize_mapped(x, asymmetric.build_colmap(ints, fp, cols), len(ints), num_fp, bits)
    for a, b in zip(got, want):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
