"""Compiler or linker flags (argument: ``compile`` / ``link``) of the module that works on torch tensors."""
import os
import sys
import sysconfig

import torch
from torch.utils import cpp_extension

if sys.argv[1] == "compile":
    includes = cpp_extension.include_paths("cuda") + [sysconfig.get_paths()["include"]]
    print("-D__HIP_PLATFORM_AMD__=1 -DUSE_ROCM=1 -DTORCH_API_INCLUDE_EXTENSION_H -D_GLIBCXX_USE_CXX11_ABI=%d "
          % int(torch._C._GLIBCXX_USE_CXX11_ABI) + " ".join("-isystem " + path for path in includes))
else:
    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    print("-L%s -lc10 -lc10_hip -ltorch_cpu -ltorch_hip -ltorch -ltorch_python -Wl,-rpath,%s" % (lib, lib))
