"""bf16 products of ragged tensors on the 256 x 256 kernel: operands copied along k into whole steps, the last tile of a dimension
moved back, the contraction in slices; the fused layer whose pass over the cotangent writes dz both ways."""
import numpy as np
import pytest

from oracle import luxlib_oracle as O
from tests.util import assert_close, dev, f64, host_inputs, kernels_of, stable_seed

pytestmark = pytest.mark.gpu

# one more and one less than a whole tile, whole tiles whose K is no whole step, short and long K (1537 x 3841 x 5001 and 1793 x 3071 x 8200: two
# slices, 1281 x 2049 x 12001: four), every layout
SHAPES = [(3841, 4095, 1001, "tt"), (3584, 4096, 1001, "nn"), (2047, 6401, 1090, "tn"), (7681, 7937, 450, "nt"), (1537, 3841, 5001, "nt"),
          (1793, 3071, 8200, "tn"), (1281, 2049, 12001, "tt")]


@pytest.mark.parametrize("M,N,K,layout", SHAPES)
def test_products(gpu, M, N, K, layout):
    tA, tB = layout[0] == "t", layout[1] == "t"
    rng = np.random.default_rng(stable_seed("large ragged", M, N, K))
    A, B, bias = host_inputs("bf16", rng.standard_normal((K, M) if tA else (M, K), np.float32), rng.standard_normal((N, K) if tB else (K, N), np.float32),
                             rng.standard_normal(M, np.float32))
    dA, dB, db = (dev(gpu, a, "bf16") for a in (A, B, bias))
    got = gpu.matmul(dA, dB, db, tA, tB).to_numpy()
    kernels = kernels_of(gpu, lambda: gpu.matmul(dA, dB, db, tA, tB))
    assert "dense_gemm_kernel<bf16>" in kernels and ("slices_reduce_kernel" in kernels) == (K > 5000)
    f32 = lambda a: np.asarray(f64(a), np.float32)          # products of bf16 are exact, sums over K in fp32: 1e-6 of a result
    want = (f32(A).T if tA else f32(A)) @ (f32(B).T if tB else f32(B)) + f32(bias)[:, None]
    assert_close(got, want, "bf16", f"{M} x {N} x {K} {layout}")
    np.testing.assert_array_equal(got, gpu.matmul(dA, dB, db, tA, tB).to_numpy())


def test_zeros_behind_k_are_not_multiplied(gpu):
    """What lies behind an operand's rows does not reach the sums: both copies are zero there, and an infinity in the last k of one operand
    reaches its row only."""
    M, N, K = 4000, 4001, 1001
    A, B = np.ones((M, K), np.float32), np.ones((K, N), np.float32)
    A[3, K - 1] = np.inf
    got = gpu.matmul(dev(gpu, A, "bf16"), dev(gpu, B, "bf16")).to_numpy()
    want = np.full((M, N), float(K))
    want[3] = np.inf
    want = np.asarray(f64(O.round_to_bf16(want.astype(np.float32))))
    np.testing.assert_array_equal(got, want)


# batch, inputs and outputs ragged; outputs whole (dz read where it lies), identity (dz is the cotangent itself); an activation that needs y
@pytest.mark.parametrize("act,M,K,N", [("gelu", 3301, 3075, 3067), ("tanh", 3328, 3075, 3067), ("identity", 3264, 3136, 3067),
                                         ("identity", 3301, 3072, 3072)])
def test_layer(gpu, act, M, K, N):
    rng = np.random.default_rng(stable_seed("large ragged layer", act, M))
    W, x, b, delta = host_inputs("bf16", rng.standard_normal((M, K), np.float32) / np.sqrt(K), rng.standard_normal((K, N), np.float32),
                                 0.1 * rng.standard_normal(M, np.float32), rng.standard_normal((M, N), np.float32))
    y, back = gpu.pullback(gpu.fused_dense_bias_activation, act, *(dev(gpu, a, "bf16") for a in (W, x, b)))
    ddelta = dev(gpu, delta, "bf16")
    assert "dense_dz_kmajor_kernel" in kernels_of(gpu, lambda: back(ddelta))
    gW, gx, gb = back(ddelta)
    f32 = lambda a: np.asarray(f64(a), np.float32)
    z = f32(W) @ f32(x) + f32(b)[:, None]
    wy = O.act_value(act, f64(z))
    assert_close(y.to_numpy(), wy, "bf16", f"{act} y")
    stored = lambda a: f64(O.round_to_bf16(np.asarray(a, np.float32)))
    dz = O.grad_activation(f64(delta), stored(wy), act, stored(z))
    assert_close(gb.to_numpy().reshape(-1), dz.sum(1), "bf16", f"{act} db")
    dz = np.asarray(stored(dz), np.float32)
    assert_close(gW.to_numpy(), dz @ f32(x).T, "bf16", f"{act} dW")
    assert_close(gx.to_numpy(), f32(W).T @ dz, "bf16", f"{act} dx")


class TallView:
    """The first `rows` rows of a bf16 matrix of 2^22 + 8 rows and 256 columns: 256 of its columns are 2^31 bytes apart and more, which the
    256 x 256 kernel does not address."""
    ld = (1 << 22) + 8

    def __init__(self, gpu, values):                        # values: rows x 256
        self.memory = gpu.DeviceArray((self.ld, values.shape[1]), "bf16")
        self.ptr = self.memory.ptr
        packed = dev(gpu, values, "bf16")
        for j in range(values.shape[1]):
            gpu._lib.call("luxhip_memcpy_d2d", self.ptr + 2 * j * self.ld, packed.ptr + 2 * j * values.shape[0], 2 * values.shape[0], gpu.current_stream())
        gpu._lib.call("luxhip_stream_synchronize", gpu.current_stream())       # before `packed` is given back


def test_rows_of_a_tall_matrix(gpu):
    """An operand whose leading dimension the 256 x 256 kernel does not take: copied for the product and for the layer's input gradient."""
    rng = np.random.default_rng(stable_seed("tall"))
    K, M, N, columns = 4096, 256, 5001, 12001
    W, x, B, delta = host_inputs("bf16", rng.standard_normal((K, M), np.float32), rng.standard_normal((M, columns), np.float32),
                                 rng.standard_normal((K, N), np.float32), rng.standard_normal((K, columns), np.float32))
    tall, dB, got = TallView(gpu, W), dev(gpu, B, "bf16"), gpu.DeviceArray((M, N), "bf16")
    product = lambda: gpu._lib.call("luxhip_matmul", gpu.current_stream(), dB.code, 1, 0, M, N, K, tall.ptr, tall.ld, dB.ptr, K, None, got.ptr, M)
    assert {"kmajor_rows_kernel", "dense_gemm_kernel<bf16>"} <= set(kernels_of(gpu, product))
    assert_close(got.to_numpy(), W.T @ B, "bf16", "W' B")
    dx, dd = dev(gpu, x, "bf16"), dev(gpu, delta, "bf16")
    gW, gx, gb = (gpu.DeviceArray(s, "bf16") for s in ((K, M), (M, columns), (K,)))
    layer = lambda: gpu._lib.call("luxhip_fused_dense_bwd", gpu.current_stream(), dd.code, 0, K, M, columns, dd.ptr, None, None, tall.ptr, tall.ld, dx.ptr, M,
                                  None, gW.ptr, gx.ptr, gb.ptr)
    assert {"kmajor_rows_kernel", "dense_gemm_kernel<bf16>"} <= set(kernels_of(gpu, layer))
    assert_close(gW.to_numpy(), delta @ x.T, "bf16", "dW")
    assert_close(gx.to_numpy(), W.T @ delta, "bf16", "dx")
    assert_close(gb.to_numpy(), f64(delta).sum(1), "bf16", "db")
