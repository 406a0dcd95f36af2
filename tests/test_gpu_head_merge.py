"""GPU parity of the LM head's merge of the screen's candidate lists: up to 16
chunks of 64 entries (one per wave) and beyond (folded), one worker."""
import pytest

from tests.test_gpu_head import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [16384, 16640])      # 64 lists of 16 entries: 16 chunks; 65: 17
def test_merge_chunks(gpu, V):
    run(V, 64, 31, nt=1, cand=16, dup=True)
