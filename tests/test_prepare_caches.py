"""The caches of a source preparation share one allocation and are otherwise tensors of their own: one may be changed in
place, also by something that requires a gradient, without a word to the others."""
import pytest
import torch

from mkx.prepare import _layer_caches


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("shape", [(3, 5, 2, 64), (5, 2, 64)])
def test_caches_are_tensors_of_their_own(shape, grad):
    with torch.set_grad_enabled(grad):
        kv = torch.empty(2 * 4 * shape[0], *shape[1:], dtype=torch.bfloat16)
        layers = _layer_caches(kv, 4)
    flat = [t for pair in zip(*layers) for t in pair]  # K of every layer, then V
    assert len(layers) == 4 and len(flat) == 8
    for i, t in enumerate(flat):
        assert t.shape == shape and t.is_contiguous() and t.dtype == torch.bfloat16
        assert t.data_ptr() == kv.data_ptr() + i * t.numel() * 2
        t.fill_(float(i))
    (k0, v0), (k1, _) = layers[0], layers[1]
    versions = [t._version for t in flat[1:]]
    with torch.enable_grad():
        k0.add_(torch.ones(shape, dtype=torch.bfloat16, requires_grad=True))
    assert k0.requires_grad and not any(t.requires_grad for t in flat[1:])
    assert [t._version for t in flat[1:]] == versions
    k1.detach_()
    assert bool((k0 == 1).all() and (k1 == 1).all() and (v0 == 4).all())
