"""The split product for weight gradients (long K, small C): edges of its 16 x
16 tiles and of K's sixteenths, aligned and unaligned rows, both sides of the
rule that chooses it."""
import numpy as np
import pytest


def _bf16(x):
    b = np.asarray(x, dtype=np.float32).view(np.uint32).astype(np.uint64)
    b = (b + 0x7FFF + ((b >> 16) & 1)) >> 16 << 16
    return b.astype(np.uint32).view(np.float32).astype(np.float64)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 1, 256), (16, 16, 512), (17, 15, 515), (135, 128, 4096),
                                   (128, 46, 4099), (33, 129, 255), (1024, 512, 300),
                                   (1030, 512, 300)])
def test_long_products_match_numpy(M, N, K):
    """Tolerance: an FP32 sum of K exact products, at most K additions deep,
    errs by at most K 2^-24 sum |a b| (the products of two BF16 values are
    exact), alpha, beta and the final sum by three more roundings."""
    from pypde_amd.learned import Dev, gemm
    rng = np.random.default_rng(M + N + K)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = rng.standard_normal((N, K)).astype(np.float32)
    C0 = rng.standard_normal((M, N)).astype(np.float32)
    Ct = Dev.from_numpy(C0)
    gemm(Dev.from_numpy(A), Dev.from_numpy(B), Ct, transB=True, alpha=0.5, beta=2.0)
    a, b = _bf16(A), _bf16(B)
    want = 0.5 * (a @ b.T) + 2.0 * C0
    bound = 2.0 ** -24 * ((0.5 * K + 2) * (np.abs(a) @ np.abs(b).T) + 6.0 * np.abs(C0))
    got = Ct.numpy()
    assert np.all(np.abs(got - want) <= bound)
    again = Dev.from_numpy(C0)
    gemm(Dev.from_numpy(A), Dev.from_numpy(B), again, transB=True, alpha=0.5, beta=2.0)
    assert np.array_equal(again.numpy(), got)   # the same sums in the same order
