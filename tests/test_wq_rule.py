"""Which packed-weight products of few rows cut K over the waves of a workgroup (ops/csrc/gemm_wq.hip wq_slices_pay): sizes on either side of
its lines, by the measurements beside it."""
import pytest

from vllm_distributed_amd.ops import native as N


@pytest.mark.parametrize("M,n,k,bits,pays", [(16, 2048, 4096, 4, True), (8, 2048, 6144, 4, True), (16, 2048, 6144, 4, False), (16, 1280, 8192, 4, False),
                                             (4, 1280, 8192, 8, False), (16, 2560, 8192, 8, False), (9, 1024, 4096, 8, True), (1, 256, 14336, 4, False),
                                             (16, 8192, 8192, 4, True), (10, 8192, 14336, 4, True), (2, 8192, 28672, 4, False),
                                             (12, 8192, 28672, 8, True), (13, 8192, 28672, 8, False), (8, 4096, 28672, 8, False),
                                             (16, 10240, 8192, 4, False), (16, 14336, 8192, 4, True), (16, 28672, 4096, 4, False),
                                             (9, 28672, 4096, 8, True), (4, 57344, 8192, 8, True), (5, 57344, 8192, 8, False), (1, 57344, 8192, 4, False),
                                             (17, 4096, 4096, 4, False)])
def test_rule(M, n, k, bits, pays):
    assert N.lib().vda_wq_slices_pay(M, n, k, bits, 128, 0) == pays


def test_where_the_other_kernel_cannot_cut_k():
    pay = N.lib().vda_wq_slices_pay
    assert pay(16, 1281, 8192, 4, 128, 1) and pay(10, 1281, 28672, 4, 128, 1) and not pay(13, 1281, 28672, 8, 128, 1)


@pytest.mark.parametrize("M,n,k,pays", [(10, 1280, 8192, True), (16, 1280, 8192, False), (10, 8192, 14336, True), (8, 8192, 28672, True), (8, 4096, 28672, False),
                                        (8, 10240, 8192, True), (16, 14336, 8192, True), (8, 28672, 8192, True), (16, 28672, 8192, False)])
def test_rule_of_groups_of_64(M, n, k, pays):
    assert N.lib().vda_wq_slices_pay(M, n, k, 4, 64, 0) == pays


@pytest.mark.parametrize("M,n,k,bits,parts", [(13, 10240, 8192, 4, 6), (64, 10240, 8192, 8, 6), (65, 10240, 8192, 4, 3), (13, 5120, 5120, 4, 5), (65, 5120, 13824, 4, 6),
                                              (13, 21760, 4096, 8, 3), (13, 21888, 4096, 8, 1), (32, 28672, 4096, 4, 1), (33, 28672, 4096, 4, 2),
                                              (32, 28672, 5248, 4, 2), (64, 32768, 4096, 8, 1), (13, 32896, 4096, 8, 2), (13, 49024, 4096, 4, 2),
                                              (13, 49152, 4096, 4, 1), (128, 24448, 4096, 4, 1), (128, 24576, 4096, 4, 1), (16, 256, 512, 4, 1)])
def test_parts_of_one_round(M, n, k, bits, parts):
    assert N.lib().vda_wq_parts(M, n, k, bits) == parts
