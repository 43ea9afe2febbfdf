"""The text reader's device memory follows the rows it is asked for: a few rows
in front of many blank lines are read in little of it."""
import gc

import numpy as np
import pytest

import topk_amd

pytestmark = pytest.mark.gpu


def test_few_rows_of_many_lines(gpu, tmp_path):
    import torch
    lines = 16_000_000
    p = tmp_path / "blank.csv"
    p.write_bytes(b"1.5,2\n3,4.25\n" + b"\n" * lines + b"5,6\n")
    gc.collect()
    torch.cuda.empty_cache()
    free, _ = torch.cuda.mem_get_info()
    # the text and 8 bytes a line (144 MB), not 16 more a line
    hold = torch.empty(free - (260 << 20), dtype=torch.uint8, device="cuda")
    rep = topk_amd.read_csv(str(p), n=2, d=2)
    del hold
    torch.cuda.empty_cache()
    x = rep[0] if isinstance(rep, tuple) else rep
    assert np.array_equal(np.asarray(x).reshape(2, 2), [[1.5, 3.0], [2.0, 4.25]])
    whole = topk_amd.read_csv(str(p))
    x = whole[0] if isinstance(whole, tuple) else whole
    assert np.array_equal(np.asarray(x).reshape(2, 3), [[1.5, 3.0, 5.0], [2.0, 4.25, 6.0]])
