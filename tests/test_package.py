"""Loading the package: models without the tensor side's extension, and that extension never from another source."""
import os
import shutil
import subprocess
import sys
import sysconfig

import deepj_amd
from deepj_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _copy(tmp_path):
    package = tmp_path / "deepj_amd"
    os.makedirs(package / "csrc")
    for name in os.listdir(build.HERE):
        if name.endswith(".py"):
            shutil.copy(os.path.join(build.HERE, name), package)
    shutil.copy(os.path.join(build.CSRC, "graph_core.cpp"), package / "csrc")
    return package


def _run(tmp_path, program, **env):
    return subprocess.run([sys.executable, "-c", program], cwd=tmp_path, env={**os.environ, "DEEPJ_HIP_LIBRARY": deepj_amd.LIB_PATH, **env},
                          capture_output=True, text=True, timeout=120)


def test_models_need_no_compiler(tmp_path):
    """Where the extension is not built and cannot be, all but the tensor side is there, and that says what is missing."""
    _copy(tmp_path)
    r = _run(tmp_path, "import deepj_amd as d; from deepj_amd import build, fused, models, persistence, LlamaConfig; d.HipNative.q8Floats(64, 2); "
                       "assert 'Tensor' in dir(d) and set(d.__all__) <= set(dir(d))\n"
                       "try:\n    d.Tensor\nexcept RuntimeError as e:\n    print(e)", PATH=str(tmp_path))
    assert r.returncode == 0 and "no g++" in r.stdout, r.stdout + r.stderr


def test_the_extension_is_that_of_its_source(tmp_path):
    package = _copy(tmp_path)
    program = "import deepj_amd as d; d.Tensor(1, 2); print(d.compute_graph._graph_core.__file__)"
    (package / "_graph_core.so").write_text("an extension of some other version")
    files = []
    for _ in range(2):
        r = _run(tmp_path, program)
        assert r.returncode == 0, r.stderr
        files.append(r.stdout.strip())
        with open(package / "csrc" / "graph_core.cpp", "a") as f:
            f.write("// changed\n")
    assert files[0] != files[1] and all(f.endswith(sysconfig.get_config_var("EXT_SUFFIX")) for f in files)
    assert [f for f in os.listdir(package) if f.endswith(".so")] == [os.path.basename(files[1])]


def test_the_tensor_side_is_where_it_was():
    import deepj_amd.tensor
    assert deepj_amd.Tensor is deepj_amd.tensor.Tensor and deepj_amd.compute_graph.GpuBuffer is deepj_amd.GpuBuffer
    assert deepj_amd.hip_backend.HipBackend is deepj_amd.HipBackend
    namespace = {}
    exec("from deepj_amd import *", namespace)
    assert set(deepj_amd.__all__) <= set(namespace)
