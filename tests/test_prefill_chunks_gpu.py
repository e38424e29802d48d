"""A prompt's hidden rows and logits have the same bits however it is cut into
chunks of whole 64-token DeltaNet chunks (GPU): the products' rows do not depend on
the call, the DeltaNet restarts at every 64 tokens, and the attention's sums at
every unit of keys."""

import numpy as np
import pytest
import torch

from qvex.model import Config, random_model

DEV = "cuda:0"


def bits(t):
    return t.contiguous().view(torch.int16)


@pytest.mark.gpu
@pytest.mark.parametrize("full_width", [False, True])
def test_prompt_bits_do_not_depend_on_the_chunks(full_width):
    cfg = Config.qwen35_9b() if full_width else Config.tiny(layers=4, vocab=4096)
    cfg.num_hidden_layers = 4
    m = random_model(cfg, seed=81, device=DEV, max_context=2048)
    n = 1344
    ids = torch.from_numpy(np.random.default_rng(82).integers(0, cfg.vocab_size, n).astype(np.int32)).reshape(1, -1)

    def run(chunk):
        cache, rows = m.make_cache(), []
        for i in range(0, n, chunk):
            logits, hidden = m(ids[:, i:i + chunk], cache, return_hidden=True)
            rows.append(hidden[0].clone())
        return torch.cat(rows), logits.clone()

    hidden, logits = run(512)
    for chunk in (64, 128, 256, 320):
        h, lg = run(chunk)
        differ = (bits(h) != bits(hidden)).sum().item()
        assert differ == 0, f"chunks of {chunk}: {differ} of {h.numel()} hidden values differ"
        assert torch.equal(lg, logits), chunk
