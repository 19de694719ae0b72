#!/bin/bash
# Builds glq_amd/libglq_hip.so for gfx950 (cross-compiles without a GPU) and glq_amd/_glq_host.so, the
# native host path in front of it.  Extra arguments go to every hipcc line.
set -e
here="$(cd "$(dirname "$0")" && pwd)"
out="$here/../libglq_hip.so"
obj="$(mktemp -d)"
trap 'rm -rf "$obj"' EXIT
python3 - "$obj/host.args" <<'PY'
import sys, sysconfig, torch, torch.utils.cpp_extension as c
lib = c.library_paths()[0]
with open(sys.argv[1], "w") as f:
    f.write(" ".join(["-I" + p for p in c.include_paths() + [sysconfig.get_paths()["include"], "/opt/rocm/include"]] +
                     ["-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI, "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
                      "-L" + lib, "-Wl,-rpath," + lib, "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch", "-ltorch_python"]))
PY
pids=()
g++ -O2 -std=c++17 -fPIC -shared -fvisibility=hidden -Wall "$here/host.cpp" $(cat "$obj/host.args") -o "$here/../_glq_host.so" &
pids+=($!)
for f in "$here"/*.hip; do
    /opt/rocm/bin/hipcc --offload-arch=gfx950 -O3 -std=c++17 -fPIC -c \
        -Xclang -target-feature -Xclang -packed-fp32-ops \
        -Wall -Wno-unused-function "$@" "$f" -o "$obj/$(basename "$f" .hip).o" &
    pids+=($!)
done
failed=0
for p in "${pids[@]}"; do wait "$p" || failed=1; done
[ $failed = 0 ]
/opt/rocm/bin/hipcc --offload-arch=gfx950 -fPIC -shared "$obj"/*.o -o "$out"
echo "built $out and _glq_host.so"
