"""Prints what calls.cpp is compiled and linked with against the torch of this interpreter, as the compiler reads it from a file."""
import os
import sysconfig

import torch

root = os.path.dirname(torch.__file__)
print(" ".join([
    f'-DSB_TORCH_VERSION=\\"{torch.__version__}\\"',
    f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
    f"-isystem {root}/include -isystem {root}/include/torch/csrc/api/include -isystem {sysconfig.get_paths()['include']}",
    f"-L{root}/lib -ltorch_python -ltorch_cpu -lc10"]))
