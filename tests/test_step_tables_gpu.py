"""The tables of a step's rows and query tiles, beyond 64 rows written on the device (csrc/mixers_ops.hip: step_tables_kernel): whole numbers, equal to those made entry by entry."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens,q_tile", [([1], 128), ([128, 129, 127, 1], 128), ([1] * 300, 128), ([7, 8192, 1, 256, 255], 128), ([5, 64, 65], 32), ([3, 1, 2], 1), ([64], 32), ([65], 32), ([1] * 64, 128), ([1] * 65, 128)])
def test_rows_and_tiles(lens, q_tile):
    from gbx_lm_amd.batching import StepBatch
    first = [(i * 37) % 11 for i in range(len(lens))]
    slot = list(range(len(lens)))[::-1]
    for device in ("cuda:0", "cpu"):
        b = StepBatch.build(slot, first, lens, device, q_tile)
        starts = [sum(lens[:i]) for i in range(len(lens))]
        assert b.total == sum(lens) and b.q_tile == q_tile
        assert b.seq.tolist() == [[s, p, n, r] for s, p, n, r in zip(slot, first, lens, starts)]
        assert b.tok.tolist() == [[i, p + j] for i, (p, n) in enumerate(zip(first, lens)) for j in range(n)]
        assert b.tiles.tolist() == [[i, t] for i, n in enumerate(lens) for t in range(0, n, q_tile)]
        assert all(t.dtype == torch.int32 and t.is_contiguous() for t in (b.seq, b.tok, b.tiles))


def test_a_sequence_without_rows_is_refused():
    from gbx_lm_amd.batching import StepBatch
    with pytest.raises(ValueError):
        StepBatch.build([0, 1], [0, 0], [3, 0], "cuda:0")
