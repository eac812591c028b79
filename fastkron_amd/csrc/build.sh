#!/bin/bash
# Builds libFastKron.so (the C-ABI library) for gfx950 with hipcc, in-tree.
#   fastkron_amd/csrc/build.sh           (takes no arguments: the kernels have no build-time switches)
set -euo pipefail
if (( $# )); then echo "build.sh takes no arguments" >&2; exit 2; fi
HERE="$(cd "$(dirname "${BASH_SOURCE[0]}")" && pwd)"
OUT="$HERE/../lib"
OBJ="$HERE/../lib/obj"
mkdir -p "$OUT" "$OBJ"
HIPCC="${HIPCC:-/opt/rocm/bin/hipcc}"
# -packed-fp32-ops is switched off: hipcc must not form v_pk_*_f32 from scalar float code.
FLAGS=(-O3 -std=c++17 -fPIC --offload-arch=gfx950 -Xclang -target-feature -Xclang -packed-fp32-ops
       -Wall -Wno-unused-function -Wno-unused-value -Wno-unused-result -Wno-unused-command-line-argument -I"$HERE/../../include")
SRCS=("$HERE"/api.cpp "$HERE"/handle.cpp "$HERE"/kernel_db.cpp "$HERE"/autotuner.cpp "$HERE"/gradient.cpp "$HERE"/static_scratch.hip "$HERE"/kernels/*.hip)
pids=()
objs=()
for s in "${SRCS[@]}"; do
  o="$OBJ/$(basename "$s").o"
  objs+=("$o")
  "$HIPCC" "${FLAGS[@]}" -x hip -c "$s" -o "$o" &
  pids+=($!)
  if (( ${#pids[@]} >= 8 )); then wait "${pids[0]}"; pids=("${pids[@]:1}"); fi
done
for p in "${pids[@]}"; do wait "$p"; done
"$HIPCC" -shared -fPIC --offload-arch=gfx950 -o "$OUT/libFastKron.so" "${objs[@]}"
echo "built $OUT/libFastKron.so"
# the PyTorch front end's host path: host code only, against the headers of the PyTorch that runs it
read -r -a TORCH < <(python3 - <<'PY'
import os, sysconfig, torch
from torch.utils import cpp_extension
print(*(f"-isystem {p}" for p in cpp_extension.include_paths() + [sysconfig.get_paths()["include"]]),
      f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f"-L{os.path.join(os.path.dirname(torch.__file__), 'lib')}")
PY
)
g++ -O2 -std=c++17 -fPIC -shared -fvisibility=hidden -Wall -I"$HERE/../../include" "$HERE/frontend.cpp" -o "$OUT/_frontend.so" \
    "${TORCH[@]}" -ltorch_python -ltorch_cpu -ltorch -lc10
echo "built $OUT/_frontend.so"
