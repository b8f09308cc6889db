"""The DAG words that ``ResidentScenes`` takes, on the CPU: what the conversion kernels, which
read consecutive words from a pointer, are given."""

import warnings

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


@pytest.mark.parametrize("keep_words", [False, True])
@pytest.mark.parametrize("source", ["frozen", "mapped", "bytes"])
def test_read_only_words_load_without_a_warning(source, keep_words, tmp_path):
    """Words of a frozen array, a memory-mapped file and a byte string, as an asset's reader
    holds them."""
    words = np.array([0xFF << 55 | 1, *[9] * 8, 1 << 63 | 3 << 16 | 0x2E66], np.uint64)
    if source == "mapped":
        words.tofile(tmp_path / "words")
        given = np.memmap(tmp_path / "words", np.uint64, "r")
    else:
        given = np.frombuffer(words.tobytes(), np.uint64)
        if source == "frozen":
            given = words.copy()
            given.setflags(write=False)
    assert not given.flags.writeable
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        got = multiscene.ResidentScenes([(given, [0.0] * 3, [1.0] * 3)], "cpu", keep_words=keep_words)
        upload = got._words(got.pool if keep_words else np.ascontiguousarray(given))
    assert got.relaid_ok and got.word_counts == [10]
    assert np.array_equal(upload.numpy().view(np.uint64), words)
