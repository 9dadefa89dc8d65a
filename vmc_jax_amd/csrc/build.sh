#!/bin/bash
# Builds libjvmc_hip.so for gfx950 in-tree (next to this script's package): the
# sources side by side (one hipcc each, at most as many as there are CPUs, 16
# at the most), then one link.
set -euo pipefail
here="$(cd "$(dirname "$0")" && pwd)"
out="${JV_OUT:-$here/../libjvmc_hip.so}"
HIPCC="${HIPCC:-/opt/rocm/bin/hipcc}"
flags=(${JV_EXTRA_FLAGS:-} -O3 -std=c++17 -fPIC --offload-arch=gfx950 -mcode-object-version=5
       -Xclang -target-feature -Xclang -packed-fp32-ops
       -Wno-unused-result -Wno-unused-parameter)
# the longest compilations first
srcs=(sampler nets eloc batch symrbm linalg tridiag core sym qapply dc chol gram_mixed)
work="$(mktemp -d)"
trap 'rm -rf "$work"' EXIT
jobs="$(nproc)"
printf '%s\n' "${srcs[@]}" | xargs -P "$((jobs < 16 ? jobs : 16))" -I{} \
  "$HIPCC" "${flags[@]}" -c "$here/{}.hip" -o "$work/{}.o"
objs=()
for s in "${srcs[@]}"; do objs+=("$work/$s.o"); done
"$HIPCC" -shared --offload-arch=gfx950 "${objs[@]}" -o "$out.tmp" -L/opt/rocm/lib -lrocsolver -lrocblas
mv "$out.tmp" "$out"
echo "built $out"
