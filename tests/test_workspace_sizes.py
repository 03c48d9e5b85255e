"""The *_workspace_size queries (host code, no GPU): a workspace sized for the longest chunk or the widest step holds
every shorter one, so a caller may size once."""
import os

import pytest

SHAPES = [(256, 8, 4096, 2048), (256, 8, 256, 128), (1024, 1, 256, 128), (1024, 16, 256, 128), (8, 2, 256, 512),
          (40, 6, 768, 384), (3, 1, 256, 128)]
# every length to 1400 (past the 640 tokens up to which the router's logits come as partial sums), and both sides of
# the 24 routes a slot at which the GEMMs' tiles change
TOKENS = lambda E, k: sorted(set(range(1, 1401)) | set(range(max(1, 24 * E // k - 40), 24 * E // k + 40)))


@pytest.fixture(scope="module")
def lib():
    from mimo_stream import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("libmimo_moe.so not built")
    return _lib.load()


@pytest.mark.parametrize("E,k,H,I", SHAPES)
def test_prefill_need_never_falls(lib, E, k, H, I):
    queries = {"block": lambda T: lib.mimo_moe_prefill_block_workspace_size(T, E, k, E, H, I),
               "layer": lambda T: lib.mimo_moe_layer_prefill_workspace_size(T, E, k, E, H, I),
               "experts": lambda T: lib.mimo_moe_prefill_workspace_size(T, k, E, H, I),
               "dispatch": lambda T: lib.mimo_prefill_dispatch_workspace_size(T, k, E)}
    for name, size in queries.items():
        need = [size(T) for T in TOKENS(E, k)]
        falls = [(T, a, b) for T, a, b in zip(TOKENS(E, k), need, need[1:]) if b < a]
        assert not falls, f"{name}: first fall after {falls[0]}"


@pytest.mark.parametrize("E,k,H,I", [s for s in SHAPES if s[1] <= 8])
def test_decode_need_never_falls(lib, E, k, H, I):
    for size in (lib.mimo_moe_decode_workspace_size, lib.mimo_moe_layer_decode_workspace_size):
        need = [size(M, E, k, H, I) for M in range(1, 9)]
        assert need == sorted(need)
