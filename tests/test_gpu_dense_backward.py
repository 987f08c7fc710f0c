"""coral_amd_nn_gemm16 and coral_amd_nn_gemm_gelu_bwd against the calls they
join, at the edges of the 64 x 64 tiles, odd leading dimensions and split K."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cl(native_lib):
    from coral_amd import closure
    return closure


def _bf16(cl, a):
    from coral_amd.devmem import DevArray
    d32, d16 = DevArray.from_numpy(a.astype(np.float32)), DevArray(a.size, "bf16")
    cl.check(cl.lib.coral_amd_nn_cast_bf16(d32.ptr, d16.ptr, a.size, None), "cast")
    return d16


@pytest.mark.parametrize("N,K", [(1, 8), (9, 9), (64, 64), (100, 40), (256, 64), (66, 33)])
@pytest.mark.parametrize("M", [1, 63, 64, 65, 200, 1024])
def test_gelu_backward_product(cl, M, N, K):
    from coral_amd.devmem import DevArray
    lib, check = cl.lib, cl.check
    rng = np.random.default_rng(M + N)
    A, B = _bf16(cl, rng.standard_normal((M, K))), _bf16(cl, rng.standard_normal((N, K)))
    Z = DevArray.from_numpy((3 * rng.standard_normal((M, N))).astype(np.float32))
    dA, d16, e16 = DevArray(M * N), DevArray(M * N, "bf16"), DevArray(M * N, "bf16")
    out = DevArray(N)
    check(lib.coral_amd_nn_gemm(0, 1, M, N, K, 1.0, A.ptr, K, 0, B.ptr, K, 0, 0.0, dA.ptr, N, 0, 1, None, 0, None), "g")
    check(lib.coral_amd_nn_gelu_bwd(Z.ptr, dA.ptr, dA.ptr, d16.ptr, M * N, None), "b")
    nw = int(lib.coral_amd_nn_gemm_gelu_bwd_work(M, N))
    work = DevArray(nw)
    check(lib.coral_amd_nn_gemm_gelu_bwd(M, N, K, A.ptr, K, B.ptr, K, Z.ptr, e16.ptr, out.ptr, work.ptr, nw, None), "f")
    assert np.array_equal(d16.numpy(), e16.numpy())   # the same arithmetic
    dz = dA.numpy().reshape(M, N).astype(np.float64)
    # FP32 sums in any order: (M - 1) roundings at most, each of eps/2 of the sum of magnitudes
    bound = max(M - 1, 1) * np.finfo(np.float32).eps / 2 * np.abs(dz).sum(axis=0) + 1e-30
    assert (np.abs(out.numpy() - dz.sum(axis=0)) <= bound).all()
    rc = lib.coral_amd_nn_gemm_gelu_bwd(M, N, K, A.ptr, K, B.ptr, K, Z.ptr, e16.ptr, out.ptr, work.ptr, nw - 1, None)
    assert rc != 0   # too little work space is refused


@pytest.mark.parametrize("M,N,K,batch", [(1, 1, 8, 1), (65, 9, 40, 3), (64, 64, 32, 2), (130, 36, 72, 2),
                                         (64, 32, 4096, 1)])
def test_product_with_bf16_copy(cl, M, N, K, batch):
    from coral_amd.devmem import DevArray
    lib, check = cl.lib, cl.check
    rng = np.random.default_rng(M + K)
    A, B = _bf16(cl, rng.standard_normal((batch, M, K))), _bf16(cl, rng.standard_normal((batch, K, N)))
    C0 = rng.standard_normal(batch * M * N).astype(np.float32)
    C1, C2, h1, h2 = DevArray.from_numpy(C0), DevArray.from_numpy(C0), DevArray(C0.size, "bf16"), DevArray(C0.size, "bf16")
    nw = int(lib.coral_amd_nn_gemm_work(M, N, K, batch))
    work = DevArray(max(nw, 1))
    args = (0, 0, M, N, K, 0.5, A.ptr, K, M * K, B.ptr, N, K * N, 1.0)
    check(lib.coral_amd_nn_gemm(*args, C1.ptr, N, M * N, batch, work.ptr, nw, None), "g")
    check(lib.coral_amd_nn_cast_bf16(C1.ptr, h1.ptr, C1.n, None), "c")
    check(lib.coral_amd_nn_gemm16(*args, C2.ptr, N, M * N, batch, work.ptr, nw, h2.ptr, None), "g16")
    assert np.array_equal(C1.numpy(), C2.numpy()) and np.array_equal(h1.numpy(), h2.numpy())
