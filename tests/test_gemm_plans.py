"""Which GEMM kernel a decode projection takes (ops/gemm.py), without a GPU: the plans that tables and timing leave."""
import pytest
import torch

from kubernetes_gpu_cluster_amd.ops import gemm

M, N, K = 32, 256, 128


@pytest.fixture
def plans(monkeypatch):
    """One weight, and a K9m tile that takes it as it is."""
    monkeypatch.setattr(gemm, "_dg_info", lambda cfg: (64, 64, False))
    gemm.clear_plan()
    yield [torch.zeros(N, K)]
    gemm.clear_plan()


SKINNY = {"plain": gemm._plan, "silu": gemm._plan_silu}


@pytest.mark.parametrize("kind", ["plain", "silu", "tail", "qkv"])
def test_entries_of_a_table_take_the_place_of_skinny_plans(plans, kind):
    """The skinny kernels' plans are asked first: an entry beside one was reported as chosen and had no effect."""
    if kind in SKINNY:
        SKINNY[kind][M, N, K] = (2, 1, 4, False)
    gemm._dg_table[M, N, K, kind] = (2, 1)
    res = {}
    gemm._tune_dgemm(plans, N, K, [M], 0.97, 3, res, kind)
    assert res[M, N, K, kind][0] == gemm.dgemm_plan()[M, N, K, kind] == (2, 1)
    assert not any((M, N, K) in p for p in SKINNY.values())


@pytest.mark.parametrize("kind", sorted(SKINNY))
def test_entries_without_a_kernel_leave_skinny_plans(plans, kind):
    SKINNY[kind][M, N, K] = (2, 1, 4, False)
    gemm._dg_table[M, N, K, kind] = None
    res = {}
    gemm._tune_dgemm(plans, N, K, [M], 0.97, 3, res, kind)
    assert res[M, N, K, kind][0] is None and not gemm.dgemm_plan() and (M, N, K) in SKINNY[kind]


def test_the_residual_sum_that_is_rounded_once_stays(plans, monkeypatch):
    """SK_ACC_NORM adds fp32 sums to the residual, the consumer of K9m's slices sums rounded to 16 bits: where the first
    was chosen neither a table nor timing puts the second in its place."""
    gemm._plan_accnorm[M, N, K] = (2, 1, 4, False)
    gemm._dg_table[M, N, K, "tail"] = (2, 1)
    monkeypatch.setattr(gemm, "_time", lambda *a: pytest.fail("timed"))
    for m in (M, M + 16):
        gemm._plan_accnorm[m, N, K] = (2, 1, 4, False)
    res = {}
    gemm._tune_dgemm(plans, N, K, [M, M + 16], 0.97, 3, res, "tail")
    assert not res and not gemm.dgemm_plan() and (M, N, K) in gemm.accnorm_plan()
