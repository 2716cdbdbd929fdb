"""Rows moved in place along the permutation's cycles (tables of 512 MiB on, or 1 GiB with rows
of more than 1 KiB; rows of 256 to 4096 bytes): regular permutations
whose cycles hold no leader or one only, random ones, row widths at the edges of the lane groups, a last block that is partial."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def permutation(kind, n):
    i = torch.arange(n, device=DEV)
    if kind == "identity":
        return i
    if kind == "reversal":  # n / 2 cycles of two
        return n - 1 - i
    if kind == "pairs":
        return torch.where((i ^ 1) < n, i ^ 1, i)
    if kind == "shift":  # one cycle through neighbours
        return (i + 1) % n
    if kind == "stride":  # cycles that visit one position in every 16
        return (i + 16) % n
    if kind == "triples":  # cycles of three far apart
        third = n // 3
        p = i.clone()
        p[:third * 3] = (i[:third * 3] + third) % (third * 3)
        return p
    return torch.randperm(n, generator=torch.Generator(device=DEV).manual_seed(n), device=DEV)


@pytest.mark.parametrize("kind", ["identity", "reversal", "pairs", "shift", "stride", "triples", "random"])
@pytest.mark.parametrize("words", [16, 17, 25, 33, 64, 65, 129, 256])
def test_shuffle_in_place(pbg, kind, words):
    n = ((512 if words <= 64 else 1024) << 20) // (16 * words) + 21
    print("cycles", kind, words, n, flush=True)
    t = torch.arange(n * words * 4, dtype=torch.int32, device=DEV).view(n, words * 4).view(torch.float32)
    perm = permutation(kind, n)
    want = torch.empty_like(t)
    want[perm] = t
    pbg.native.shuffle_rows(t, perm)
    assert torch.equal(t.view(torch.int32), want.view(torch.int32))


def test_out_of_range_entry_is_refused(pbg):
    n = (512 << 20) // 400 + 21
    t = torch.zeros(n, 100, device=DEV)
    for at, value in ((0, n), (n - 1, -1), (n // 2, 2**40)):
        perm = permutation("random", n)
        perm[at] = value
        print("out of range", at, value, flush=True)
        with pytest.raises(Exception):
            pbg.native.shuffle_rows(t, perm)
