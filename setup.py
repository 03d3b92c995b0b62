"""Build the in-tree HIP extension for gfx950 (MI355X).

    PYTORCH_ROCM_ARCH=gfx950 python setup.py build_ext --inplace

The resulting deepspeed_amd/ops/_C*.so is git-ignored but ships to the GPU
box with the repo snapshot.
"""

import importlib.util
import os

from setuptools import setup

os.environ.setdefault("PYTORCH_ROCM_ARCH", "gfx950")

from torch.utils.cpp_extension import (BuildExtension, CUDAExtension,  # noqa: E402
                                       ROCM_HOME)

OPS = os.path.join("deepspeed_amd", "ops")
CSRC = os.path.join(OPS, "csrc")

DEVICE_FLAGS = ["-O3", "-std=c++17", "--offload-arch=gfx950",
                "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
# The source whose kernels name accumulation registers, and how many these are: the
# build ends where the compiler's assembly does not go with it.
NAMING, KERNELS = os.path.join(CSRC, "tile_linear.hip"), 19


def _named_registers():
    path = os.path.join(OPS, "named_registers.py")    # without the package
    spec = importlib.util.spec_from_file_location("named_registers", path)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


class Build(BuildExtension):
    def build_extensions(self):
        look = _named_registers()
        hipcc = os.path.join(ROCM_HOME, "bin", "hipcc") if ROCM_HOME else "hipcc"
        assembly = look.assembly_of(NAMING, DEVICE_FLAGS, hipcc)
        try:
            super().build_extensions()
            look.check(assembly, NAMING, KERNELS)
        finally:
            assembly.close()


ext = CUDAExtension(
    name="deepspeed_amd.ops._C",
    sources=[
        os.path.join(CSRC, "bindings.cpp"),
        os.path.join(CSRC, "cpu_adam.cpp"),
        os.path.join(CSRC, "aio.cpp"),
        os.path.join(CSRC, "shm_comm.cpp"),
        os.path.join(CSRC, "step_plan.cpp"),
        os.path.join(CSRC, "adam.hip"),
        os.path.join(CSRC, "optim.hip"),
        os.path.join(CSRC, "grad_norm.hip"),
        os.path.join(CSRC, "fp_quant.hip"),
        os.path.join(CSRC, "transpose.hip"),
        os.path.join(CSRC, "softmax_dropout.hip"),
        os.path.join(CSRC, "paged_attention.hip"),
        os.path.join(CSRC, "rows_linear.hip"),
        os.path.join(CSRC, "tile_linear.hip"),
        os.path.join(CSRC, "quantize.hip"),
        os.path.join(CSRC, "attention.hip"),
        os.path.join(CSRC, "cross_entropy.hip"),
        os.path.join(CSRC, "norms.hip"),
        os.path.join(CSRC, "rope.hip"),
        os.path.join(CSRC, "swiglu.hip"),
        os.path.join(CSRC, "spatial.hip"),
        os.path.join(CSRC, "token_ops.hip"),
        os.path.join(CSRC, "embedding.hip"),
    ],
    extra_compile_args={
        "cxx": ["-O3", "-std=c++17", "-fopenmp", "-mavx2", "-mfma"],
        "nvcc": DEVICE_FLAGS,
    },
    extra_link_args=["-fopenmp"],
)

setup(
    name="deepspeed_amd",
    version="0.1.0",
    packages=["deepspeed_amd"],
    ext_modules=[ext],
    cmdclass={"build_ext": Build.with_options(use_ninja=True)},
)
