"""Device memory of a predictor handle, most of it the training work (inference handles hold it too).

Per fine-grid point: activations 200 bytes, the weight gradients' channel-major copies 720 (in the data
gradients' place) and 164, the layers' gradients or their partial sums 246: 1340 with the head's arrays;
1450 are allowed, and 8 MB for parameters and rounding.  (One buffer for each took 1940.)"""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(96, 96, 96), (60, 92, 100)])
def test_predictor_memory(n):
    import torch

    from salmon2_amd.unet import UNet

    print(f"[gpu] predictor memory {n}", flush=True)
    UNet(8, 8, 8).close()
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    u = UNet(*n)
    used = free0 - torch.cuda.mem_get_info()[0]
    u.close()
    points = n[0] * n[1] * n[2]
    print(f"[memory] predictor {n}: {used / points:.0f} bytes per point", flush=True)
    assert used <= 1450 * points + (8 << 20)
