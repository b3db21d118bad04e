"""Small host programs against the library's own functions, for rules that the C ABI does not show.  No GPU needed."""
import os
import subprocess

from cudabert_amd import build


def compile_program(source: str, folder) -> str:
    """Path of the program compiled from `source` in `folder`."""
    from cudabert_amd import pybert                      # noqa: F401  (raises if the library is not built)
    (folder / "main.hip").write_text(source)
    exe = str(folder / "main")
    flags = build.COMMON_FLAGS + build.DEVICE_FLAGS
    for cmd in (["-c", str(folder / "main.hip"), "-o", exe + ".o", "-I", build.CSRC] + flags,
                [exe + ".o", "-o", exe, build.LIB, "-Wl,-rpath," + build.HERE, "--hip-link"] + build.DEVICE_FLAGS):
        subprocess.run([build.hipcc()] + cmd, check=True, capture_output=True)
    return exe


def lines(exe: str, *args, **env) -> list:
    out = subprocess.run([exe] + [str(a) for a in args], check=True, capture_output=True, text=True,
                         env=dict(os.environ, HIP_VISIBLE_DEVICES="", **env))
    return out.stdout.splitlines()
