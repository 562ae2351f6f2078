"""Host-side rules of the kernels (csrc/*.h without device code) compiled for the CPU, so that tests
can ask them: `rules(tmp_dir, header, body)` builds the extern "C" functions of `body`."""
import ctypes
import subprocess

from conftest import PKG


def rules(tmp, header, body):
    src, lib = tmp / "rules.cpp", tmp / "rules.so"
    src.write_text(f'#include "{header}"\nextern "C" {{\n{body}\n}}\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{PKG / 'csrc'}", str(src),
                    "-o", str(lib)], check=True, capture_output=True, text=True)
    return ctypes.CDLL(str(lib))
