"""Tests of the fused pipeline written for its stage launches, run on them: their small
meshes take resident launches by default, where graphs, per-node geometry, tile options,
walks and the probe launch of each step have no part.  NW_RESIDENT=0 keeps every solver
made below to stage launches."""
import pytest
import test_gpu_batch as batch
import test_gpu_probes as probes
import test_gpu_solver as solver

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def stage_launches(monkeypatch):
    monkeypatch.setenv("NW_RESIDENT", "0")


@pytest.mark.parametrize("name", sorted(solver.CASES))
def test_fp64_matches_oracle(name):
    solver.test_fp64_matches_oracle(name, "fused")


@pytest.mark.parametrize("precision", ["fp32", "fp32_k64"])
@pytest.mark.parametrize("name", ["pec_tm110_p4", "periodic_jitter_p7"])
def test_fp32_matches_oracle(name, precision):
    solver.test_fp32_matches_oracle(name, precision)


@pytest.mark.parametrize("name", ["pec_tm110_p4", "media_pec_p5", "sheared_n8"])
def test_affine_records_equal_per_node_geometry(name, monkeypatch):
    solver.test_affine_records_equal_per_node_geometry(name, monkeypatch)


def test_graph_and_stream_paths_are_bitwise_equal_and_deterministic():
    solver.test_graph_and_stream_paths_are_bitwise_equal_and_deterministic()


@pytest.mark.parametrize("name", ["media_pec_p5", "periodic_jitter_p7"])
def test_segment_choices_give_the_same_bits(name):
    solver.test_segment_choices_give_the_same_bits(name)


def test_tune_between_runs_keeps_the_state():
    solver.test_tune_between_runs_keeps_the_state()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_cpp_reference_kats(precision):
    solver.test_cpp_reference_kats_on_device(precision)


@pytest.mark.parametrize("precision,use_graph", [("fp64", True), ("fp32", True), ("fp64", False)])
def test_probe_records_match_host_record_each_step(precision, use_graph):
    probes.test_probe_records_match_host_record_each_step("fused", precision, use_graph)


def test_probe_history_overflow_is_an_error():
    probes.test_probe_history_overflow_is_an_error()


def test_case_launches_output_intervals_as_one_run():
    probes.test_case_launches_output_intervals_as_one_run()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_batch_equals_single_runs_and_oracle(precision):
    batch.test_batch_equals_single_runs_and_oracle(precision)
