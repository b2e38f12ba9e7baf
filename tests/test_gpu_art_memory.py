"""init_diffuse_gpu on a device whose free memory does not hold the default
batch's accumulator slices: a smaller batch, with the same rates; a batch that the
caller asked for is refused as before."""
import numpy as np
import pytest
import torch

from argot_amd import art as A
from argot_amd import ic

pytestmark = pytest.mark.gpu

GIB = 1 << 30


def test_default_batch_fits_the_free_memory(require_gpu):
    w = ic.art128(seed=15, n=128)
    st = A.DiffuseStep(w)          # 256 directions: 8 GiB of slices
    st.step()
    want = st.rates()
    st.close()
    print("diffuse transfer with 5.5 GiB free", flush=True)
    torch.cuda.empty_cache()
    free, _ = torch.cuda.mem_get_info()
    held = torch.empty(free - 11 * GIB // 2, dtype=torch.uint8, device="cuda")
    try:
        st = A.DiffuseStep(w)
        st.step()
        got = st.rates()
        st.close()
        with pytest.raises(RuntimeError):
            A.DiffuseStep(w, batch=256)
    finally:
        del held
        torch.cuda.empty_cache()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
