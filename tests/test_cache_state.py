"""BitKVCache's bookkeeping that needs no GPU."""
import io

import torch


def test_a_cache_saved_without_device_lengths_still_decodes():
    """A saved cache is rebuilt from its attributes: one from before the device length arrays has none."""
    from bitladder_amd import BitKVCache
    cache = BitKVCache(2, 1, 256, device="cpu")
    cache.packed_len, cache.res_len = [128, 0], [5, 7]
    state = dict(vars(cache))
    state.pop("_published", None)
    old = BitKVCache.__new__(BitKVCache)
    file = io.BytesIO()
    torch.save(state, file)
    file.seek(0)
    old.__dict__.update(torch.load(file, weights_only=False))
    packed, window = old._device_lengths()
    assert packed.tolist() == [128, 0] and window.tolist() == [5, 7]
