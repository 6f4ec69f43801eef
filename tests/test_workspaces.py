"""Workspace sizes of the prepared MoE layer (host arithmetic of the library, no GPU): a
workspace for T tokens serves every smaller T, whatever plan those take."""
import random

import pytest


@pytest.mark.parametrize("seed", range(4))
def test_moe_prepared_workspace_grows_with_the_tokens(seed):
    import gaje_hip
    size = gaje_hip.ops.moe_ffn_prepared_workspace
    rng = random.Random(seed)
    shapes = [(1536, 4096, 8), (1344, 1248, 8), (2816, 1504, 3), (2112, 160, 15), (64, 96, 16)]
    shapes += [(32 * int(2 ** rng.uniform(0, 7)), 32 * int(2 ** rng.uniform(0, 8)), rng.randint(2, 16)) for _ in range(8)]
    for h, ffn, experts in shapes:
        last = 0
        for tokens in range(1, 800):
            now = size(tokens, h, ffn, experts)
            assert now >= last, (h, ffn, experts, tokens)
            last = now
