#!/bin/bash
# Optional AddressSanitizer HOST build of libp3v.so + the launcher check that runs without a GPU.
# The device code is compiled as usual (GPU ASan / xnack+ objects are not available on this pool: -fno-gpu-sanitize);
# only the host side -- the extern "C" launchers, their argument validation, the tuning table -- is instrumented.
#   tools/asan_host_build.sh            -> build/libp3v_asan.so, build/asan_host_check, runs the check
set -e
cd "$(dirname "$0")/.."
mkdir -p build
SRC=phi-3-vision-mlx_amd/csrc
OBJ=build/asan_obj; mkdir -p $OBJ
PIDS=()
for f in $SRC/p3v_*.hip; do                                       # every translation unit, as the library
  hipcc --offload-arch=gfx950 -O1 -g -Xclang -target-feature -Xclang -packed-fp32-ops -std=c++17 -fPIC -fsanitize=address -fno-gpu-sanitize -Wno-unused-result -c $f -o $OBJ/$(basename $f .hip).o & PIDS+=($!)
  while [ "$(jobs -rp | wc -l)" -ge 8 ]; do wait -n || exit 1; done
done
for p in "${PIDS[@]}"; do wait "$p" || exit 1; done
hipcc --offload-arch=gfx950 -g -fPIC -fsanitize=address -fno-gpu-sanitize -shared-libsan -shared $(for f in $SRC/p3v_*.hip; do echo $OBJ/$(basename $f .hip).o; done) -o build/libp3v_asan.so
/opt/rocm/lib/llvm/bin/clang++ -O1 -g -std=c++17 -fsanitize=address -shared-libsan tools/asan_host_check.cpp -o build/asan_host_check \
  -Lbuild -lp3v_asan -Wl,-rpath,'$ORIGIN' -Wl,-rpath,/opt/rocm/lib
ASAN_OPTIONS=detect_leaks=0:abort_on_error=1 LD_LIBRARY_PATH=build:$(dirname $(/opt/rocm/lib/llvm/bin/clang++ -print-file-name=libclang_rt.asan-x86_64.so)):/opt/rocm/lib ./build/asan_host_check
