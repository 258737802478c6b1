"""Token-to-expert alignment at the edges of the kernel that holds all ids in registers: lists that end inside a lane's four ids, a wavefront's and a
workgroup's run and behind the longest one it takes, ids that start off a 16-byte boundary, more experts than workgroups, experts without a token
and ids of no expert.  Whole numbers, equal element for element to an independent stable sort."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def stable_sort(ids: torch.Tensor, experts: int, block: int, slots: int, blocks: int):
    rows, owners, at = torch.full((slots,), ids.numel(), dtype=torch.int32), torch.zeros(blocks, dtype=torch.int32), 0
    for e in range(experts):
        mine = (ids == e).nonzero()[:, 0].int()
        room = (mine.numel() + block - 1) // block * block
        rows[at:at + mine.numel()] = mine
        owners[at // block:(at + room) // block] = e
        at += room
    return rows, owners, at


@pytest.mark.parametrize("experts,block", [(8, 16), (128, 64), (257, 48), (1024, 16), (1, 128)])
@pytest.mark.parametrize("numel,shift", [(1, 0), (255, 0), (1024, 0), (1025, 1), (2048, 0), (2049, 0), (4808, 0), (8193, 3), (16384, 0), (16385, 0),
                                         (32769, 2), (65536, 0), (65537, 0), (70001, 1)])
def test_align_held_edges(numel, shift, experts, block):
    from vllm_amd._custom_ops import moe_align_block_size
    gen = torch.Generator().manual_seed(numel + experts)
    # -1: of another rank; the upper half of the experts gets few or no ids
    ids = (torch.rand(numel + shift, generator=gen) ** 2 * (experts + 1)).int() - 1
    assert int(ids.max()) < experts
    slots = numel + experts * (block - 1)
    blocks = (slots + block - 1) // block
    rows, owners, total = (torch.full((n,), -7, dtype=torch.int32, device="cuda") for n in (slots, blocks, 1))
    moe_align_block_size(ids.cuda()[shift:], experts, block, rows, owners, total)
    want = stable_sort(ids[shift:], experts, block, slots, blocks)
    assert total.item() == want[2]
    assert torch.equal(rows.cpu(), want[0])
    assert torch.equal(owners.cpu(), want[1])
