"""The fused prefill GEMM's launch against its work queues (host arithmetic in the library, no GPU): a block runs one
tile of its XCD's queue, so a queue with more tiles than the launch gives its XCD blocks would leave tiles out.

The plan kernel's dealing is restated here: an expert's pairs in items of 64, its items in the fewest groups of at most
dsh_pf_unit_items, the groups and the shared expert's items ranked by cost and dealt to 8 queues in snake order."""
import random

import pytest


def longest_queue(pairs, T, H, I, SI, unit):
    """Tiles of the longest queue for an expert's pair counts."""
    ngu_r, ngu_s, ndn = I // 128, SI // 128, H // 256
    cost_r = ngu_r * (H // 128) + ndn * (I // 128)
    cost_s = ngu_s * (H // 128) + ndn * (SI // 128)
    units = [(cost_s, ngu_s + ndn)] * -(-T // 64)
    for n in pairs:
        items = -(-n // 64)
        groups = -(-items // unit)
        for g in range(groups):
            size = items // groups + (g < items % groups)
            units.append((size * cost_r, size * (ngu_r + ndn)))
    units.sort(key=lambda u: -u[0])
    tiles = [0] * 8
    for rank, (_, n) in enumerate(units):
        pos = rank % 16
        tiles[pos if pos < 8 else 15 - pos] += n
    return max(tiles)


def draw_pairs(rng, T, E, K, repeated):
    """Pairs per expert of T tokens, the first of which list expert 0 K times, the others K experts that lean."""
    pairs = [0] * E
    pairs[0] = repeated * K
    lean = [rng.random() ** 4 + 1e-6 for _ in range(E)]
    for _ in range(T - repeated):
        for e in sorted(range(E), key=lambda e: rng.random() ** (1 / lean[e]))[E - K:]:
            pairs[e] += 1
    return pairs


@pytest.mark.parametrize("H,I,SI,E,K", [(1280, 896, 1792, 64, 6), (256, 128, 256, 16, 6), (512, 256, 512, 32, 6),
                                        (2048, 1024, 128, 64, 8), (256, 128, 2048, 8, 8), (768, 2048, 256, 64, 1)])
def test_no_queue_is_longer_than_its_blocks(lib, H, I, SI, E, K):
    L = lib.load()
    rng = random.Random(H + I + E)
    for T in (1, 20, 63, 64, 65, 66, 100, 128, 129, 200, 449, 512, 513, 662, 900):
        unit, blocks = L.dsh_pf_unit_items(T), L.dsh_pf_queue_blocks(H, I, SI, E, K, T)
        assert 1 <= unit <= 8 and blocks > 0
        for repeated in sorted({0, T // 8, T // 2, (7 * T) // 8, T}):
            pairs = draw_pairs(rng, T, E, K, repeated)
            assert longest_queue(pairs, T, H, I, SI, unit) <= blocks, (T, repeated, pairs)
        # one pair in each of many experts, the rest in one
        pairs = [1] * E
        pairs[0] = max(T * K - E + 1, 0)
        assert longest_queue(pairs, T, H, I, SI, unit) <= blocks, T


def test_ordinary_tokens_keep_an_expert_in_one_unit(lib):
    """At most one pair per token: an expert's items (up to 8) stay together, so its weights are streamed once."""
    L = lib.load()
    for T in (1, 64, 65, 320, 512, 513, 3001):
        assert L.dsh_pf_unit_items(T) == min(8, -(-T // 64))


def test_queue_blocks_refuse_bad_shapes(lib):
    L = lib.load()
    assert L.dsh_pf_queue_blocks(256, 64, 128, 16, 6, 10) == -1
    assert L.dsh_pf_queue_blocks(256, 128, 256, 16, 6, 0) == -1
