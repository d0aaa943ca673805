"""Partial last tiles of the tile selection, whose waves hold unequal shares of the columns: the
bounded top-k of bfloat16 rows against the stable-sort oracle, bit-exact."""

import pytest
import torch

from oracle.topk import topk as oracle_topk

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("values", ["spread", "tied", "masked"])
@pytest.mark.parametrize("block", [1024, 4096, 16384])
def test_partial_last_tile(block, values):
    """Last tiles of 1 column to a chunk and a bit: one wave holding most of the columns, waves
    without any, shares at the edge of a wave's 128-entry run."""

    from sonic_sampler.interface import UnshardedBoundedTopK

    g = torch.Generator().manual_seed(block)

    for rest in (1, 60, 128, 129, 255, 256, 257, 300, 511, 512, 513, 700, 1023, 1025, 1281, 2049):

        if rest >= block:

            continue

        vocab = block + rest
        x = torch.randn(5, vocab, generator=g) * 3

        if values == "tied":

            x = torch.randint(-2, 3, (5, vocab), generator=g).float()

        if values == "masked":

            # few finite values, some of them only in the last tile
            keep = torch.rand(5, vocab, generator=g) < torch.tensor([0.002, 0.02, 0.1, 0.3, 0.9])[:, None]
            keep[:, block:] = torch.rand(5, rest, generator=g) < 0.5
            x = x.masked_fill(~keep, -float("inf"))

        # the last tile holds more of the top 128 than any other
        x[::2, block:] += 4.0
        x = x.to(torch.bfloat16)

        for k in (1, 32, 128):

            print(f"block {block} rest {rest} k {k} {values}", flush=True)
            topk = UnshardedBoundedTopK.initialize(vocab_size=vocab, batch_size=5, k=k, block_size=block, device=DEV)
            got_values, got = topk(x.to(DEV))
            want_values, want = oracle_topk(x, k)
            assert torch.equal(got.cpu(), want)
            assert torch.equal(got_values.cpu(), want_values)
