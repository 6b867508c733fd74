"""Re-indexing of Jacobian rows by a table, for every form of the kernel: vector and single floats, four output rows to a thread and
one, groups of slots; the sums are formed in slot order, so the bits are those of the same additions one after another."""

import pytest
import torch

from folx_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('k_in,k_out,n_slots,B,S_outer,S_inner', [
    (2, 1, 1, 1, 1, 1), (3, 3, 5, 7, 3, 4), (3, 4, 4, 5, 3, 4), (3, 5, 3, 5, 3, 3), (1, 7, 1, 257, 1, 1), (4, 9, 2, 33, 4, 8),
    (3, 8, 9, 20, 11, 1), (2, 3, 4, 3, 2, 6), (3, 66, 1, 64, 5, 64), (0, 5, 1, 3, 2, 4), (3, 6, 0, 3, 2, 4),
    (2, 5, 2, 524281, 1, 3), (1, 1, 1, 600000, 1, 4),                       # more walkers than 8 x 65535
])
def test_gather_rows_in_slot_order(k_in, k_out, n_slots, B, S_outer, S_inner):
    print(f'case gather k {k_in} -> {k_out} slots {n_slots} B={B} S={S_outer} x {S_inner}', flush=True)
    g = torch.Generator().manual_seed(k_out * 100 + n_slots)
    data = torch.randn(k_in, B, S_outer, S_inner, generator=g)
    take = torch.randint(-1, k_in, (k_out, n_slots, S_outer), generator=g, dtype=torch.int32)
    want = torch.zeros(k_out, B, S_outer, S_inner)
    for t in range(k_out):
        for s in range(n_slots):
            for o in range(S_outer):
                if take[t, s, o] >= 0:
                    want[t, :, o] += data[take[t, s, o], :, o]
    flat = data.reshape(k_in, B, S_outer * S_inner).cuda()
    got = K.gather_rows(flat, take.cuda(), k_out, n_slots, B, S_outer, S_inner)
    assert torch.equal(got.cpu().reshape(want.shape), want)
    # data that starts off a 16-byte boundary takes the single-float form
    shifted = torch.empty(flat.numel() + 1, device='cuda')[1:].copy_(flat.reshape(-1)).reshape(flat.shape)
    assert torch.equal(K.gather_rows(shifted, take.cuda(), k_out, n_slots, B, S_outer, S_inner), got)
