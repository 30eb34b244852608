"""GPU parity of the kernels whose sizes a small call decides, against the
oracle: the arithmetic encoder's load groups."""
import numpy as np
import pytest

from conftest import MODEL_PATH

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd():
    import czip_amd
    if czip_amd.device_count() < 1:
        pytest.fail("no HIP device visible")
    return czip_amd


@pytest.fixture(scope="module")
def pair(amd, orc):
    return amd.Model(amd.ModelWeights(MODEL_PATH)), orc.Model.from_file(MODEL_PATH)


@pytest.mark.parametrize("chunk", [1, 7, 8, 9, 16, 65])
def test_encoder_chunk_lengths(pair, chunk):
    """Chunk lengths around the encoder's groups of eight intervals, with a
    ragged last chunk; uniform ids, so that symbols of 20 to 30 bits (several
    words' worth of pending bits among them) are common."""
    gm, om = pair
    n = 67 * chunk + (chunk + 1) // 2
    toks = np.random.default_rng(chunk).integers(0, 1024, n).astype(np.uint32)
    assert gm.compress_chunks(toks, chunk) == om.compress_many(toks, chunk, threads=4)
