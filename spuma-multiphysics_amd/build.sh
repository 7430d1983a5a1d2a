#!/usr/bin/env bash
# Builds lib/libreactiveTransport.so (HIP, gfx950) from csrc/.
# Rounding policy: IEEE FP64, no contraction (-ffp-contract=off), no fast-math;
# search.hip (the FP32 candidate search only) adds -freciprocal-math -fapprox-func.
# Stack slots are not shared: where the lanes of a wave take both sides of a
# branch around calls, the compiler keeps the scalar registers that one side
# saves (stores of all 64 lanes) in slots that lanes of the other side still use.
# lanes.hip, two.hip: the registers that hold saved scalars are allocated without
# splitting (-wwm-regalloc=basic).  A split's copy runs for all 64 lanes, and
# the ordinary allocation puts single lanes' moves and spills inside it (up to
# 42 instructions in the FP64 flash's frozen solve), which overwrote other
# lanes' values: a batch of binary cells, one per lane, read a wild pointer.
# Constants stay in the loops that use them there (-disable-machine-licm):
# hoisted, they are most of the scalars to save (of two.hip's 19,000 saves
# 8,600 are left), and with it a batch of 80,000 binary cells takes 1,516 ms
# instead of 1,798.
# The other files' kernels have no such copy with anything inside it; a change
# to the code around them can bring one (tests/test_whole_wave_registers.py
# looks the built library over).
set -euo pipefail
here="$(cd -- "$(dirname -- "${BASH_SOURCE[0]}")" && pwd)"
hipcc="${HIPCC:-/opt/rocm/bin/hipcc}"
mkdir -p "$here/lib" "$here/_build"
flags=(--offload-arch=gfx950 -O3 -std=c++17 -fPIC -ffp-contract=off -fno-fast-math
       -Xclang -target-feature -Xclang -packed-fp32-ops
       -mllvm -no-stack-slot-sharing
       -I"$here/../include" -Wall -Wno-unused-result)
objs=()
pids=()
for src in "$here"/csrc/*.hip; do
  obj="$here/_build/$(basename "${src%.hip}").o"
  rm -f "$obj"
  extra=()
  # the FP32 candidate search may use approximate reciprocals and transcendentals
  if [ "$(basename "$src")" = "search.hip" ]; then extra=(-freciprocal-math -fapprox-func); fi
  if [ "$(basename "$src")" = "lanes.hip" ] || [ "$(basename "$src")" = "two.hip" ]; then extra=(-mllvm -wwm-regalloc=basic -mllvm -disable-machine-licm); fi
  "$hipcc" "${flags[@]}" "${extra[@]}" -c "$src" -o "$obj" 2> >(grep -v "packed-fp32-ops" >&2) &
  objs+=("$obj")
  pids+=("$!")
done
failed=0
for pid in "${pids[@]}"; do
  wait "$pid" || failed=1
done
if [ "$failed" -ne 0 ]; then
  echo "build.sh: a HIP compile failed" >&2
  exit 1
fi
"$hipcc" --offload-arch=gfx950 -shared -fPIC "${objs[@]}" -o "$here/lib/libreactiveTransport.so.tmp"
mv "$here/lib/libreactiveTransport.so.tmp" "$here/lib/libreactiveTransport.so"
