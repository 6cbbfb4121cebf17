"""CPU: which weight gradients take the library's own kernel (csrc/kd_torch.cpp, weight_grad_pays)."""
import pytest

from kerneldev_amd import _lib


@pytest.mark.parametrize("M,N,K,own", [
    # us on an MI355X, own / torch's product
    (2048, 768, 768, True),      # 15.4 / 18.4
    (128, 2048, 768, True),      # 10.5 / 17.9
    (768, 2048, 768, True),      # 16.1 / 18.2
    (1536, 2048, 768, False),    # 20.3 / 18.6
    (2048, 2048, 768, False),    # 22.3 / 19.9
    (16384, 2048, 768, True),    # 63 / 132
    (1024, 2048, 1024, False),   # 19.4 / 18.4
    (2048, 2048, 1024, False),   # 22.8 / 20.2
    (5000, 2048, 1024, True),    # 31.5 / 47.0
    (2560, 2048, 512, False),    # 20.3 / 19.4
    (2560, 512, 2048, True),     # 17.9 / 19.3
    (2048, 4096, 256, False),    # 20.9 / 18.9
    (1024, 1448, 1448, False),   # 19.8 / 18.7
    (4096, 64, 32768, False),    # 56 / 52
    (1024, 8, 262144, False),    # 107 / 97
    (16384, 2048, 1032, False),  # past the widest dW measured
])
def test_rule(M, N, K, own):
    assert _lib.native().weight_grad_pays(M, N, K) is own
