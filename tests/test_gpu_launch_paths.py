"""The launches around the projections: what an operation publishes to the host, and the small
kernels a layer's launch sequence is made of, at the edges of their ranges."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbytes", [0, 4, 1028, 65536])
def test_publish_brings_results_and_status_to_the_host(gpu, nbytes):
    from yvex_amd import load_library
    lib = load_library()
    host = C.c_void_p()
    assert lib.yvex_hip_host_alloc(C.byref(host), C.c_uint64(64 + 65536)) == 0
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    data = torch.arange(max(nbytes // 4, 1), dtype=torch.int32, device=gpu) * 3 + 1
    status = torch.tensor([2], dtype=torch.int32, device=gpu)
    seen = C.c_int(-1)

    def publish(count, clear, sequence):
        return lib.yvex_hip_publish(C.c_void_p(data.data_ptr()), C.c_uint64(count), C.c_void_p(status.data_ptr()),
                                    C.c_int(clear), host, C.c_uint32(sequence), stream)
    try:
        for sequence, clear, want in ((1, 0, 2), (2, 1, 2), (3, 1, 0)):      # kept, then cleared, then clear
            assert publish(nbytes, clear, sequence) == 0
            assert lib.yvex_hip_await(host, C.c_uint32(sequence), C.byref(seen), stream) == 0
            assert seen.value == want
            got = np.ctypeslib.as_array((C.c_int32 * (nbytes // 4)).from_address(host.value + 64))
            assert np.array_equal(got, data.cpu().numpy()[:nbytes // 4])
        assert publish(65540, 1, 4) == -7 and publish(2, 1, 4) == -10
    finally:
        torch.cuda.synchronize()
        lib.yvex_hip_host_free(host)
