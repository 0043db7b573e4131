#!/bin/bash
# Builds libsslm_hip.so in place (gfx950).  Usage: superslm_amd/build.sh
# Any compile or link failure exits non-zero; objects are rebuilt from scratch every time so a
# stale object can never be linked into the library.
set -euo pipefail
cd "$(dirname "$0")"
FLAGS="-O3 -std=c++17 -fPIC --offload-arch=gfx950 -Xclang -target-feature -Xclang -packed-fp32-ops"
rm -rf _build
mkdir -p _build
compile() {
  local src=$1 obj=$2 log
  log=$(mktemp)
  if ! hipcc $FLAGS -c "$src" -o "$obj" >"$log" 2>&1; then
    cat "$log" >&2
    rm -f "$log"
    echo "build.sh: compiling $src failed" >&2
    exit 1
  fi
  # The host pass warns that it does not know the packed-fp32 feature: harmless, filtered out.
  grep -v "packed-fp32-ops" "$log" >&2 || true
  rm -f "$log"
}
PIDS=()
OBJS=()
for src in csrc/*.hip csrc/*.cpp; do
  obj=_build/$(basename "${src%.*}").o
  OBJS+=("$obj")
  compile "$src" "$obj" &
  PIDS+=($!)
done
FAIL=0
for p in "${PIDS[@]}"; do wait "$p" || FAIL=1; done
if [ $FAIL -ne 0 ]; then
  rm -f libsslm_hip.so
  exit 1
fi
hipcc -shared -fPIC --offload-arch=gfx950 "${OBJS[@]}" -lcrypto -o libsslm_hip.so.tmp
mv libsslm_hip.so.tmp libsslm_hip.so
