"""Single-GPU stand-in for the reference's ``custom_a2a`` (layers/all_to_all.py:10-125).

The reference's operator moves rows between GPUs with Iris puts (kernels.py:21-146).  The
inter-GPU transfer is not part of a one-GPU build; what is kept is the operator's contract: the
10-argument signature, the in-place fill of ``local_pca`` / ``token_buf`` / the two completion
counters, and the returned ``token_buf``.  The sends of the other simulated ranks are supplied
through a ``SimulatedWorld``; one HIP kernel gathers the rows from all of them into place ([E_local, world, CAP, H], zero
padded), with the counts and counters.  The host waits once, for the largest count (a kernel of its own in front leaves
it in pinned memory), because an overflow raises.
"""
from __future__ import annotations

import contextlib
from typing import Dict, Optional, Tuple

import torch

from .. import _lib as L
from .. import ops
from ..utils import _assert_cuda_int32


class SimulatedWorld:
    """What every simulated source rank would send: (payload, dest_counts [W,E_l], dst_offsets [W])."""

    def __init__(self, world_size: int, rank: int = 0):
        self.world_size = int(world_size)
        self.rank = int(rank)
        self.sends: Dict[int, Tuple[torch.Tensor, torch.Tensor, torch.Tensor]] = {}

    def post(self, src: int, tokens: torch.Tensor, dest_counts: torch.Tensor, dst_offsets: torch.Tensor) -> None:
        assert 0 <= src < self.world_size
        self.sends[int(src)] = (tokens, dest_counts, dst_offsets)


_current: Optional[SimulatedWorld] = None


@contextlib.contextmanager
def simulated_world(world: SimulatedWorld):
    global _current
    prev, _current = _current, world
    try:
        yield world
    finally:
        _current = prev


class AllToAllOp(torch.autograd.Function):

    @staticmethod
    def forward(ctx, tokens, dest_counts, dst_offsets, local_pca, token_buf, counts_ready, token_sync, heap_bases,
                experts, capacity):
        """Same arguments as the reference (layers/all_to_all.py:13-46).  ``heap_bases`` is ignored."""
        _assert_cuda_int32(dest_counts, "dest_counts")
        _assert_cuda_int32(dst_offsets, "dst_offsets")
        _assert_cuda_int32(local_pca, "local_pca")
        world_size = local_pca.shape[1]
        world = _current if _current is not None else SimulatedWorld(world_size, 0)
        assert world.world_size == world_size, "simulated world size does not match local_pca"
        # the reference's assert is inverted (all_to_all.py:80); the intent is divisibility
        assert experts % world_size == 0, "EP-group size unevenly calculated."
        e_local = experts // world_size
        rank = world.rank
        world.post(rank, tokens, dest_counts, dst_offsets)

        # what each source sends to `rank`: rows [dst_offsets[rank], +sum(dest_counts[rank,:]))
        sends, shape, where = [None] * world_size, (world_size, e_local), (tokens.device, torch.int32)
        for src, (p, dc, do) in world.sends.items():
            assert p.shape[1:] == tokens.shape[1:] and dc.shape == shape and do.numel() == world_size, "sends of different shapes"
            # (as posted they are usually what the kernels read; otherwise a converted copy)
            if p.dtype != tokens.dtype or not (p.is_cuda and p.is_contiguous()):
                p = p.to(tokens.device, tokens.dtype).contiguous()
            if dc.dtype != torch.int32 or not (dc.is_cuda and dc.is_contiguous()):
                dc = dc.to(*where).contiguous()
            if do.dtype != torch.int32 or not (do.is_cuda and do.is_contiguous()):
                do = do.to(*where).contiguous()
            sends[src] = (p, dc, do)
        want = (e_local, world_size, capacity, tokens.shape[-1])
        block, most = ops.a2a_sources(sends, rank), ops.pinned_i32(2)
        fits = tuple(token_buf.shape) == want and token_buf.dtype == tokens.dtype
        ops.a2a_max_count(block, e_local, most)
        # (an exchange of one launch writes nothing if a count exceeds the capacity, and the host learns of that while the rows move;
        # of several, each launch knows its own sources' counts only, so the host looks at the largest of all first)
        if world_size > L.MOE_A2A_SOURCES:
            ops.wait_i32(most)
            fits = fits and int(most[0]) <= capacity
        try:
            if fits:
                pca = local_pca if local_pca.is_contiguous() else torch.empty_like(local_pca, memory_format=torch.contiguous_format)
                ready, sync = (t if t.dtype == torch.int32 and t.is_cuda and t.is_contiguous() else None for t in (counts_ready, token_sync))
                ops.a2a_place(block, token_buf, pca, ready, sync)
        finally:
            ops.wait_i32(most)
        over = int(most[0])
        if over > capacity:
            raise ValueError(f"capacity overflow: a (src, expert) pair sends {over} rows > CAP={capacity}")
        if not fits:
            raise ValueError(f"token_buf shape {tuple(token_buf.shape)} mismatch expected "
                             f"({e_local},{world_size},{capacity},{tokens.shape[-1]}) of {tokens.dtype}.")
        if pca is not local_pca:
            local_pca.copy_(pca)
        # completion counters in their final state: every source has signalled (all_to_all.py:59-69)
        if ready is None:
            counts_ready.fill_(world_size)
        if sync is None:
            token_sync.fill_(world_size)
        return token_buf

    @staticmethod
    def backward(ctx, *grad_outputs):
        raise NotImplementedError("Backward pass not implemented yet.")


custom_a2a = AllToAllOp.apply
