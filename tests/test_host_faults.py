"""The library's host code when something goes wrong: its objects linked against a pretended HIP runtime (tests/host/fake_hip.cpp),
so that a refused call, a failed launch or memory that runs out is seen on the CPU and nothing is done to a GPU."""
import pytest


@pytest.fixture(scope="session")
def model_file(oracle, tmp_path_factory):
    import lfm2_synth

    path = tmp_path_factory.mktemp("model") / "small.gguf"
    path.write_bytes(bytes(lfm2_synth.build(oracle, seed=5)[0]))
    return str(path)


def test_copies_out_of_range_are_refused_before_anything_is_enqueued(host_faults):
    host_faults("ranges")


def test_a_copy_that_fails_leaves_nothing_on_its_way(host_faults, model_file):
    host_faults("copies", model_file)


def test_a_prompt_that_fails_leaves_nothing_pending(host_faults, model_file):
    host_faults("prompts", model_file)


def test_no_exception_leaves_an_entry_point_when_host_memory_runs_out(host_faults, model_file):
    host_faults("memory", model_file)


def test_every_launch_of_a_model_goes_to_its_own_gpu(host_faults, model_file):
    host_faults("devices", model_file)
