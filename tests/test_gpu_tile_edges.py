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


def shifted(plane, offset, pad):
    """A copy of the bf16 [rows, n] plane whose rows start `offset` halves into their storage and
    lie n + pad apart."""

    rows, n = plane.shape
    flat = torch.full((offset + rows * (n + pad) + 8,), -7.0, dtype=plane.dtype, device=plane.device)
    view = flat[offset:].as_strided((rows, n), (n + pad, 1), offset)
    view.copy_(plane)

    return view


@pytest.mark.parametrize("offset,pad", [(1, 0), (0, 1), (3, 3), (2, 0), (0, 2)])
@pytest.mark.parametrize("block,vocab", [(1024, 2052), (2048, 9000), (4096, 8196), (8192, 33000), (16384, 50280)])
def test_rows_at_any_half_word(block, vocab, offset, pad):
    """Logit and bias rows at an odd half-word or with an odd stride take the three-dword loads; at an
    offset or pad of 2 every row still starts on a dword and takes the two-dword loads at addresses that
    8 does not divide. The same values in contiguous rows take the two-dword loads, but for drafting
    over vocab - 1 columns, whose ragged width takes the three-dword loads wherever its rows start.
    Every output of the decode step, of drafting through d2t, of the verification and of the top-k is
    the same bits."""

    from sonic_sampler.core.buffer import SamplingBuffers
    from sonic_sampler.core.flags import Flags, Indicator
    from sonic_sampler.interface import UnshardedBoundedTopK
    from sonic_sampler.interface.functional import fused_multistep, fused_singular

    rows = 6
    g = torch.Generator().manual_seed(vocab + offset)
    logits = (torch.randn(rows, vocab, generator=g) * 3).to(torch.bfloat16).to(DEV)
    buffers = SamplingBuffers.random(size=rows, timesteps=1, vocab_size=vocab, device=DEV, seed=vocab,
                                     indicators=Indicator(0x7BF), max_top_logprobs=5)
    # rows of every kind: all processors, none (the logits alone), penalties only, bias only, greedy
    kinds = [0x7BF, 0x400, 0x40E, 0x410, 0x05E, 0x4B1]
    buffers.flags = Flags.from_values(rows, 1, [Indicator(k) for k in kinds], device=torch.device(DEV))
    rep = buffers.repetition
    d2t = torch.randperm(vocab, generator=g).to(torch.int32).to(DEV)
    common = dict(
        indicators=buffers.flags.target, block_n=block, context_counts=rep.counts.context,
        repetition_penalties=rep.multiplicative, frequency_penalties=rep.frequency,
        presence_penalties=rep.presence, temperature=buffers.temperature, top_k=buffers.top_k,
        top_p=buffers.top_p, min_p=buffers.min_p, philox_seed=5)

    def outputs(x, bias):

        print(f"block {block} vocab {vocab} offset {offset} pad {pad}", flush=True)
        grammar = buffers.grammar[:, 0].as_subclass(torch.Tensor)
        one = fused_singular(x, logit_bias=bias, grammar=grammar, decode_counts=rep.counts.decode, **common)
        drafts = []

        for width in (vocab - 4, vocab - 1):

            probabilities = torch.zeros(rows, vocab, dtype=torch.bfloat16, device=DEV)
            draft = fused_singular(x[:, :width], logit_bias=bias, grammar=grammar, decode_counts=rep.counts.decode,
                                   d2t_mapping=d2t[:width], target_vocab=vocab, return_probabilities=True,
                                   draft_probabilities=probabilities, **common)
            drafts += [draft.tokens, probabilities]

        values = torch.zeros(rows, 128, device=DEV)
        indices = torch.zeros(rows, 128, dtype=torch.int32, device=DEV)
        drafted = x.float().argmax(-1).to(torch.int32)
        keep = {k: v for k, v in common.items() if k != "indicators"}
        check = fused_multistep(x.unflatten(0, (rows // 2, 2)), drafted_tokens=drafted.view(rows // 2, 2),
                                indicators=buffers.flags.target[: rows // 2].clone(), lookahead=1, logit_bias=bias,
                                decode_counts=rep.counts.decode, values=values, indices=indices,
                                uniform_noise=buffers.weights.uniform.as_subclass(torch.Tensor), **keep)
        topk = UnshardedBoundedTopK.initialize(vocab_size=vocab, batch_size=rows, k=128, block_size=block, device=DEV)
        best, columns = topk(x)

        return [t.clone() for t in (one.tokens, *drafts, check.tokens, check.offsets, indices, values, best,
                                    columns)]

    want = outputs(logits, buffers.bias)
    got = outputs(shifted(logits, offset, pad), shifted(buffers.bias, offset, pad))

    for name, a, b in zip(("decode", "drafts", "probabilities", "ragged drafts", "their probabilities", "tokens", "offsets", "indices", "values", "top-k", "columns"),
                          want, got):

        assert torch.equal(a, b), f"{name} differ between aligned rows and rows at offset {offset}, pad {pad}"


@pytest.mark.parametrize("density", [0.0005, 0.01, 0.04, 0.1, 0.3])
@pytest.mark.parametrize("block,vocab", [(1024, 3000), (2048, 8193), (4096, 9000), (8192, 33000), (16384, 40002)])
def test_count_and_bias_density(block, vocab, density, monkeypatch):
    """Rows whose counts and biases are nonzero in few columns keep them in the waves' exception
    lists, in more columns overflow the lists pass by pass: the decode step, the verification (with
    drafted history) and drafting through d2t against the oracle."""

    import test_gpu_sweep as sweep

    whole = sweep.random_host

    def thinned(slots, timesteps, vocab, seed, indicator=None, **kw):

        host = whole(slots, timesteps, vocab, seed, indicator, **kw)
        g = torch.Generator().manual_seed(seed)

        for plane in (host.repetition.counts.context, host.repetition.counts.decode, host.bias):

            plane.masked_fill_(torch.rand(plane.shape, generator=g) >= density, 0)

        return host

    monkeypatch.setattr(sweep, "random_host", thinned)
    seed = 4000 + block + int(1000 * density)
    sweep.test_sweep_autoregressive(block, vocab, "random", "spiked", seed)
    sweep.test_sweep_multistep_row_top128(block, vocab, "random", "spiked", seed)
    sweep.test_sweep_drafting_d2t(block, vocab, "sparse", "spiked", seed)
    sweep.test_sweep_drafting_d2t(block, vocab, "random", "few", seed + 1)


@pytest.mark.parametrize("density", [0.002, 0.05, 0.3, 1.0])
@pytest.mark.parametrize("block,vocab", [(2048, 8193), (4096, 9000), (8192, 33000), (16384, 40002)])
def test_drafting_with_penalties_that_only_lower(block, vocab, density, monkeypatch):
    """Drafting rows whose penalties only lower logits read their counts at the selection's survivors,
    and start the selection again where too many of those fall below its bound (dense counts, tied
    values): against the oracle, with rows at the neutral ends of the ranges and drafted history."""

    import test_gpu_sweep as sweep

    whole = sweep.random_host

    def lowering(slots, timesteps, vocab, seed, indicator=None, **kw):

        host = whole(slots, timesteps, vocab, seed, indicator & ~0x1, **kw)  # no grammar
        g = torch.Generator().manual_seed(seed)
        rep = host.repetition

        for plane in (rep.counts.context, rep.counts.decode):

            plane.masked_fill_(torch.rand(plane.shape, generator=g) >= density, 0)

        rep.multiplicative.copy_(1 + (rep.multiplicative - 1).abs())
        rep.frequency.abs_()
        rep.presence.abs_()
        rep.multiplicative[0], rep.frequency[1], rep.presence[2] = 1.0, 0.0, 0.0
        rep.multiplicative[3], rep.frequency[4] = 0.9, -0.5  # these rows cannot wait

        return host

    monkeypatch.setattr(sweep, "random_host", lowering)
    seed = 6000 + block + int(1000 * density)
    sweep.test_sweep_drafting_d2t(block, vocab, "random", "spiked", seed)
    sweep.test_sweep_drafting_d2t(block, vocab, "random", "few", seed + 1)
