"""The DAG words that ``ResidentScenes`` takes, on the CPU: what the conversion kernels, which
read consecutive words from a pointer, are given."""

import numpy as np
import pytest
import torch

from navi_amd import multiscene

WORDS = torch.arange(1, 25, dtype=torch.int64)
LAYOUTS = {
    "plain": WORDS,
    "offset": WORDS[3:],
    "strided": WORDS[::2],
    "expanded": WORDS[4].expand(7),
    "rows": WORDS.view(4, 6),
    "transposed": WORDS.view(4, 6).t(),
    "columns": WORDS.view(4, 6)[:, 1:3],
    "unsigned": WORDS.view(torch.uint64)[::3],
    "scalar": WORDS[5],
}


@pytest.mark.parametrize("name", list(LAYOUTS))
def test_tensor_words_are_consecutive(name):
    words = LAYOUTS[name]
    got = multiscene._flat_words(words)
    want = words.numpy().reshape(-1).astype(np.int64)
    assert got.dtype == torch.int64 and got.is_contiguous() and got.dim() == 1
    # as a kernel reads them: numel words from the first one's address
    flat = torch.empty(0, dtype=torch.int64).set_(got.untyped_storage(), got.storage_offset(), (want.size,), (1,))
    assert flat.tolist() == want.tolist()


@pytest.mark.parametrize("dtype", [torch.float64, torch.int32, torch.uint8])
def test_other_types_are_refused(dtype):
    with pytest.raises(TypeError, match="int64"):
        multiscene._flat_words(torch.zeros(8, dtype=dtype))
