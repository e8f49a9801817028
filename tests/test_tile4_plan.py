"""Which tiles an int4 layer GEMM of fewer rows than the 256-row tiles take: the ring of 128x128 tiles (its activation comes in 6
bits) or the register-streaming tiles (4 bits), csrc/gemm_tile4.hip."""
import pytest


# (M, out, K, bits); 256 CUs.  us per forward with register-streaming tiles / on the ring, weights warm
@pytest.mark.parametrize("M,N,K,bits", [(640, 4096, 10752, 6),     # 39.0 / 34.9
                                        (512, 5120, 13568, 6),     # 42.7 / 38.9
                                        (400, 5120, 13568, 6),     # 41.1 / 38.6
                                        (300, 8192, 7936, 6),      # 27.9 / 26.7
                                        (512, 4096, 10752, 4),     # 26.8 / 33.8
                                        (256, 5120, 13568, 4),     # 25.3 / 36.6
                                        (640, 2048, 1792, 4),      # 12.8 / 15.3
                                        (512, 4096, 3840, 4)])     # 15.9 / 19.6
def test_ring_or_register_streaming_tiles(M, N, K, bits):
    from quik_amd import _lib as L
    assert L.load().quik_tile4_activation_bits(M, N, K, 256) == bits
