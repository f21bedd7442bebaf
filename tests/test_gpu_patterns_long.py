"""Seeded BigBird masks on the GPU around the row length up to which a wave keeps its draws in LDS
(1,024 blocks), with strides that leave padding, counts past what a row holds and past a wave's lanes:
the bits of the numpy oracle."""
import sys

import numpy as np
import pytest
import torch

from oracle import seeded as osd
from sparseattentioninfer_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("align", ["trailing", "centred"])
@pytest.mark.parametrize("rows,nqb,nkb,qbo,counts", [(2, 3, 1025, 1022, [3, 70]), (1, 4, 1100, 1023, [2]), (2, 5, 17, 0, [90, 0]),
                                                     (3, 2, 2049, 2040, [1, 0, 4])])
def test_long_rows_match_the_oracle(align, rows, nqb, nkb, qbo, counts):
    print(f"[patterns] {align} rows={rows} nqb={nqb} nkb={nkb} qbo={qbo}", flush=True)
    sys.stdout.flush()
    args = dict(window=4, global_blocks=2, random_blocks=counts, seed=99, window_align=align, q_block_offset=qbo)
    got = ops.seeded_bigbird_block_mask_gpu(rows, nqb, nkb, **args)
    want = osd.seeded_bigbird_block_mask(rows, nqb, nkb, **args)
    assert torch.equal(got.cpu().bool(), torch.as_tensor(np.asarray(want)).bool())
    padded = got.as_strided((rows, nqb, got.stride(1)), got.stride())
    assert int(padded[:, :, nkb:].sum()) == 0
