"""Sample-major channel gather, row by row: exact, at sizes around a block (8
slots), a workgroup's rows and the padding."""
import ctypes as C

import numpy as np
import pytest

from hcgrid_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nchan,dtype", [(1, 1, "bf16"), (7, 3, "f16"), (8, 1, "f16"), (9, 67, "bf16"),
                                           (513, 2, "bf16"), (4099, 129, "f16"), (33, 1024, "bf16")])
def test_sample_major_rows(gpu, n, nchan, dtype):
    import torch
    capi.load()
    rng = np.random.default_rng(n + nchan)
    bits = rng.integers(0, 1 << 16, (n, nchan), dtype=np.uint16)
    perm = rng.permutation(n).astype(np.int32)
    n_pad = int(capi.load().hcg_channels_padded_len(n))
    d = lambda a: torch.as_tensor(a, device="cuda")  # noqa: E731
    v, p = d(bits.view(np.int16)), d(perm)
    out = torch.full((nchan * n_pad,), 0x7EEE, dtype=torch.int16, device="cuda")
    cnt = torch.zeros(1, dtype=torch.int32, device="cuda")
    q = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    print(f"case: n={n} nchan={nchan} {dtype}", flush=True)
    capi.call("hcg_gather_channels", n, nchan, q(p), q(v), capi.DTYPE_BF16 if dtype == "bf16" else capi.DTYPE_F16, 1,
              q(out), q(cnt), C.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    want = np.zeros((n_pad // 8, nchan, 8), dtype=np.uint16)
    i = np.arange(n)
    want[i // 8, :, i % 8] = bits[perm]
    assert np.array_equal(out.cpu().numpy().view(np.uint16), want.reshape(-1))
    field = 0x7F80 if dtype == "bf16" else 0x7C00
    assert int(cnt.item()) == int(((bits & field) == field).sum())
