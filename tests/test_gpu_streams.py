"""Memory used on a second stream: the permutation's second part is copied to the device beside the update's kernels."""

from __future__ import annotations

import pytest
import torch

from oracle import rollout as R

pytestmark = pytest.mark.gpu


def test_permutation_buffer_taken_from_memory_with_work_pending():
    """The first update allocates the permutation's device buffer.  Where the allocator hands it memory whose previous
    use is still queued on the update's stream, the copy from the second stream has to wait for that use: otherwise the
    late writes replace the copied entries.  A long queue ends in a fill of a block of the buffer's size, which is
    freed before the update."""
    from tests.parity import make_pair

    w = R.scaled(R.WORKLOADS["flat48"], num_envs=4096, steps=24, hidden_dims=[32, 32])
    _, alg, _ = make_pair(w, seed=0)
    B = 4096 * 24
    x = torch.empty(B, dtype=torch.int64, device="cuda")
    big = torch.ones(4096, 4096, device="cuda")
    torch.cuda.synchronize()
    for _ in range(60):  # (a few tens of milliseconds)
        big = torch.mm(big, big).clamp_(-1.0, 1.0)
    x.fill_(7)
    del x
    torch.manual_seed(1)
    alg.update()
    torch.cuda.synchronize()
    assert torch.equal(alg._perm_dev.cpu(), alg._perm_host)
    assert torch.equal(alg._perm_dev.sort().values.cpu(), torch.arange(B))
