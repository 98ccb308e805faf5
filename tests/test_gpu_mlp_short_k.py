"""BF16 products of more tiles than the GPU has CUs around the line between their
two K steps (64 and 128 elements), in every orientation, at the tolerance and with
the padding of the other products' edge tests."""
import pytest
import test_gpu_mlp_edges as edges

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(1101, 1031, 1), (1024, 1090, 33), (1030, 1027, 63), (1024, 1088, 64),
                                   (1089, 1026, 65), (20000, 3, 64)])
@pytest.mark.parametrize("tA", [0, 1])
@pytest.mark.parametrize("tB", [0, 1])
def test_gemm_around_the_line(tA, tB, M, N, K):
    edges.test_gemm_tiles(tA, tB, M, N, K)


@pytest.mark.parametrize("M,N,K", [(1101, 1031, 7), (1030, 1027, 64), (1089, 1026, 65)])
def test_activations_around_the_line(M, N, K):
    edges.test_products_with_activation_equal_the_separate_kernels(M, N, K)


@pytest.mark.parametrize("M,N,K", [(1101, 1031, 5), (1088, 1024, 8), (1030, 1027, 31), (1024, 1090, 32), (1089, 1026, 33),
                                   (20000, 3, 17)])
@pytest.mark.parametrize("tA", [0, 1])
@pytest.mark.parametrize("tB", [0, 1])
def test_gemm_around_the_shortest_step(tA, tB, M, N, K):
    """The line between the steps of 32 and 64; whole and ragged tiles."""
    edges.test_gemm_tiles(tA, tB, M, N, K)


@pytest.mark.parametrize("M,N,K", [(1088, 1024, 20), (1024, 1090, 32)])
def test_activations_around_the_shortest_step(M, N, K):
    edges.test_products_with_activation_equal_the_separate_kernels(M, N, K)
