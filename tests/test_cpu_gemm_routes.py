"""Which kernel the contractions over two output axes lower to (no GPU)."""
import pytest

from sanic_amd import configs
from tests import gemm_forms as G


@pytest.mark.parametrize("order", ["nk view", "kn view"])
@pytest.mark.parametrize("K,N", [(2048, 8192), (8192, 2048), (2040, 1000)])
@pytest.mark.parametrize("M", [8, 33, 40, 100, 200, 300, 500])
def test_a_weight_that_is_a_view_takes_a_kernel_at_every_row_count(M, K, N, order):
    """The few-row kernel leaves a size to the GEMM only where the GEMM takes it."""
    assert G.projection(M, K, N, order).emit(0)[0].startswith("skeleton:gemm")


@pytest.mark.parametrize("order", ["nk view", "kn view"])
@pytest.mark.parametrize("M,K,N", [(64, 64, 32), (128, 512, 128), (500, 200, 1000)])
def test_the_gemm_over_a_weight_that_is_a_view_compiles(M, K, N, order):
    """... its runs are stored bf16: one product, no lo part."""
    p = G.projection(M, K, N, order)
    assert p.emit(0)[0].startswith("skeleton:gemm[") and ",b2" not in p.emit(0)[0]
    p.precompile()


@pytest.mark.parametrize("M", [32, 40, 100, 200, 300])
def test_one_4bit_group_over_a_k_off_the_tiles_takes_a_kernel(M):
    assert configs.int4_matmul(M=M, K=1056, G=1056, N=8192).emit(0)[0].startswith("skeleton:gemm_rows")


@pytest.mark.parametrize("M,K,N", [(1000, 8192, 2048), (4100, 2048, 8192), (4099, 2048, 512)])
@pytest.mark.parametrize("kmajor", [False, True])
def test_operand_planes_past_the_static_scratch_leave_a_kernel(M, K, N, kmajor):
    """Rows whose two bf16 planes pass the 32 MiB of execute_static: the kernel without planes."""
    assert configs.rmsnorm_projection(M=M, K=K, N=N, kmajor=kmajor).emit(0)[0].startswith("skeleton:gemm_rows")


@pytest.mark.parametrize("M,K,N,order,rows", [
    (2, 32768, 16, "nk", True), (2, 131072, 16, "nk", False), (2, 131072, 64, "nk", True), (2, 262144, 64, "nk", False),
    (8, 65536, 16, "nk", True), (8, 196608, 16, "nk", False), (16, 131072, 16, "nk", True),
    (2, 32768, 32, "kn", True), (2, 131072, 32, "kn", False), (2, 65536, 64, "kn", True), (2, 131072, 64, "kn", False), (8, 196608, 32, "kn", True), (2, 196608, 4096, "nk", True),
])
def test_a_long_k_under_few_points_keeps_the_split_fold(M, K, N, order, rows):
    """Where one workgroup per column block would walk K longer than the fold that splits each point."""
    kind = G.projection(M, K, N, order).emit(0)[0]
    assert kind.startswith("skeleton:gemm_rows" if rows else "fold:split"), kind
