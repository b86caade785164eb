#!/bin/sh
# The host build of the kernels lies beside them.
exec "$(cd "$(dirname "$0")/../.." && pwd)/analog_moe_amd/csrc/emu/build.sh" "$@"
