"""The gradients that the chunked and packed functions return are dense tensors of
their own, at head dims that the kernels are built for and at those they pad."""

from __future__ import annotations

import pytest
import torch

from thundersync_amd import attention as hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [64, 100, 128, 200])
def test_gradients_are_dense(cuda, dim):
    print(f"dense gradients: head dim {dim}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(dim)

    def leaf(*shape):
        return torch.randn(*shape, generator=g, device=cuda).bfloat16().requires_grad_()

    q = leaf(1, 40, 4, dim)
    ks, vs = ([leaf(n, 2, dim) for n in (70, 40)] for _ in range(2))
    out = hip.ChunkedCausalAttention.apply(q.transpose(1, 2), dim ** -0.5, 2, True, "auto", *ks, *vs)
    grads = torch.autograd.grad(out, [q, *ks, *vs], torch.randn_like(out))
    key, value = leaf(40, 2, dim), leaf(40, 2, dim)
    lay = hip.pack_layout([15, 25], [([ks[0]], [vs[0]]), ([ks[0]], [vs[0]])])
    out = hip.PackedAttention.apply(q.transpose(1, 2), key, value, dim ** -0.5, lay,
                                    *lay.inputs([([ks[0]], [vs[0]]), ([ks[0]], [vs[0]])]))
    grads += torch.autograd.grad(out, [q, key, value, ks[0], vs[0]], torch.randn_like(out))
    for t in grads:
        assert t.is_contiguous() and t.untyped_storage().nbytes() == 2 * t.numel(), (t.shape, t.stride())


@pytest.mark.parametrize("other", [32, 96])
@pytest.mark.parametrize("which", ["key", "value"])
@pytest.mark.parametrize("packed", [False, True])
def test_another_head_dim_is_refused(cuda, packed, which, other):
    """Keys or values whose head dim is not the query's raise (they were padded or cropped to it)."""
    print(f"head dim 64 against {which} of {other}, packed: {packed}", flush=True)
    dims = {"key": 64, "value": 64, which: other}
    q = torch.zeros(1, 2, 4, 64, dtype=torch.bfloat16, device=cuda)
    k, v = (torch.zeros(4, 2, dims[n], dtype=torch.bfloat16, device=cuda) for n in ("key", "value"))
    with pytest.raises(ValueError, match="must be"):
        if packed:
            hip.PackedAttention.apply(q, k, v, 0.1, hip.pack_layout([4], [([], [])]))
        else:
            hip.ChunkedCausalAttention.apply(q, 0.1, 1, True, "auto", k, v)
