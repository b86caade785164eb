#!/bin/sh
# Host build of the kernels for CPU testing: same sources as libamoe.so, with the stand-in
# headers of this directory ahead of the HIP ones.  $1 = "asan" adds the host sanitizers.
set -e
here="$(cd "$(dirname "$0")" && pwd)"
csrc="$(dirname "$here")"
include="$(cd "$csrc/../../include" && pwd)"
CXX=/opt/rocm/llvm/bin/clang++
flags="-x c++ -std=c++20 -O1 -g -fPIC -pthread -Wno-psabi -I $here -I $include -I $csrc"
link="-shared -fPIC -pthread"
out="$here/libamoe_emu.so"
if [ "$1" = "asan" ]; then
  flags="$flags -fsanitize=address,undefined -fno-omit-frame-pointer -shared-libasan"
  link="$link -fsanitize=address,undefined -shared-libasan"
  out="$here/libamoe_emu_asan.so"
fi
objdir="$here/build${1:+_$1}"
mkdir -p "$objdir"
# one translation unit per source file, compiled side by side
pids=""
objs=""
for src in "$csrc"/*.hip; do
  obj="$objdir/$(basename "$src" .hip).o"
  objs="$objs $obj"
  $CXX $flags -c "$src" -o "$obj" &
  pids="$pids $!"
done
for pid in $pids; do wait "$pid"; done
$CXX $link $objs -o "$out"
echo "$out"
