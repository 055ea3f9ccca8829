"""Host-pointer entry points on arrays that HIP knows: pinned by the caller, or in device memory.  Both are copied
by hipMemcpy itself (csrc/zq3d_hostcopy.h); the values are those of ordinary arrays."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(5, 4, 3), (96, 80, 70)], ids=str)
@pytest.mark.parametrize("where", ["pinned", "device", "mixed"])
def test_arrays_known_to_the_runtime(where, dims):
    import zq_smokesimulation_amd as z
    from zq_smokesimulation_amd import _lib
    W, H, D = dims
    print(where, dims, flush=True)
    rng = np.random.default_rng(8)
    host = [rng.standard_normal(s, np.float32) for s in ((D, H, W + 1), (D, H + 1, W), (D + 1, H, W))]
    want = z.stages.mac_to_regular4(*host)
    out = torch.zeros(want.shape)
    arrays = [torch.from_numpy(a) for a in host] + [out]
    for n, a in enumerate(arrays):
        if where == "device":
            arrays[n] = a.cuda()
        elif where == "pinned" or n % 2:
            arrays[n] = a.pin_memory()
    torch.cuda.synchronize()
    ms = _lib.lib().ZQ3D_MACtoRegular4(*[a.data_ptr() for a in arrays], W, H, D)
    assert ms >= 0.0, _lib.lib().zq3d_last_error()
    got = arrays[3].cpu().numpy()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def test_one_array_for_temperature_and_density():
    """Attenuation3D with the same array as temperature and density: both start from its values, the density
    is stored last."""
    from zq_smokesimulation_amd import _lib
    W, H, D = 128, 100, 90
    print("one array", W, H, D, flush=True)
    rng = np.random.default_rng(9)
    u, v, w, s = (rng.standard_normal(n, np.float32) for n in ((D, H, W + 1), (D, H + 1, W), (D + 1, H, W), (D, H, W)))
    want = s * np.float32(0.25)
    occ = np.zeros((D, H, W), np.uint8)
    ptr = [a.ctypes.data for a in (u, v, w, s, s, occ)]
    ms = _lib.lib().Attenuation3D(*ptr, 1.0, 0.5, 0.25, W, H, D)
    assert ms >= 0.0, _lib.lib().zq3d_last_error()
    assert np.array_equal(s.view(np.uint32), want.view(np.uint32))
