"""CPU checks of the build's order: the C library needs hipcc alone, and a host module that does not build is an
error that leaves the library in place."""
import pytest

from r2omni_amd import build


@pytest.fixture
def dry(tmp_path, monkeypatch):
    """Compiler and linker commands write empty files under ``tmp_path``; torch's headers are missing."""
    outputs = []

    def run(cmd, verbose):
        out = cmd[cmd.index("-o") + 1]
        open(out, "w").close()
        outputs.append(out)
        return ""

    def no_torch():
        raise ImportError("No module named 'torch'")

    monkeypatch.setattr(build, "_run", run)
    monkeypatch.setattr(build, "_host_flags", no_torch)
    monkeypatch.setattr(build, "_torch_libraries", no_torch)
    monkeypatch.setattr(build, "ROOT_DIR", str(tmp_path))
    for name in ("LIB_PATH", "BENCH_LIB_PATH", "TIMELINE_LIB_PATH", "HOST_PATH"):
        monkeypatch.setattr(build, name, str(tmp_path / name))
    return tmp_path


def test_the_library_builds_without_torch(dry):
    assert build.build_library() == str(dry / "LIB_PATH")
    assert (dry / "LIB_PATH").exists() and (dry / "BENCH_LIB_PATH").exists() and (dry / "TIMELINE_LIB_PATH").exists()


def test_a_host_module_that_does_not_build_leaves_the_library(dry):
    with pytest.raises(ImportError, match="torch"):
        build.build()
    assert (dry / "LIB_PATH").exists() and not (dry / "HOST_PATH").exists()


def test_the_host_module_loads_into_this_python():
    from r2omni_amd import _lib

    assert all(callable(getattr(_lib.host(), f)) for f in ("decode_handle", "decode", "cache_build"))


def test_only_the_plain_call_asks_for_the_host_module(monkeypatch):
    """The launch arguments of rotary, graph and workspace-free calls are made without it."""
    from types import SimpleNamespace

    import torch

    from r2omni_amd import _lib
    from r2omni_amd.splitk import SplitKExecutor, SplitKWorkspace

    def missing():
        raise RuntimeError("no host module")

    class OnDevice(torch.Tensor):
        is_cuda, device = True, torch.device("cuda", 0)

    monkeypatch.setattr(_lib, "host", missing)
    f32 = torch.zeros(1)
    cache = SimpleNamespace(recent_fp_pool=SimpleNamespace(fp_k=torch.zeros(1, dtype=torch.bfloat16)), bf16_key=f32)
    ws = SplitKWorkspace(partial_max=f32, partial_sum=f32, partial_output=f32, output=f32, total_blocks=1, block_n=128,
                         hierarchical_group_blocks=64, empty_bf16=f32)
    reqs = torch.zeros(1, dtype=torch.int64).as_subclass(OnDevice)
    ex = SplitKExecutor(caches=[cache], workspace=ws, reqs=reqs, items=f32, group_begin=f32, n_items=1, num_query_heads=2,
                        num_key_value_heads=1)
    assert ex._static_params().batch == 1
    with pytest.raises(RuntimeError, match="no host module"):
        ex(f32)
