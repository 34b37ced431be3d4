#!/bin/bash
# Probe builds of the 256-row prefill kernel with compile-time ablations (no GPU needed):
#   tools/fa_stamps.sh 0 12 2 31   ->  vllm_amd/csrc/libvllm_amd_probe_abl<N>.so
# then on the GPU: VLLM_AMD_LIB=vllm_amd/csrc/libvllm_amd_probe_abl12.so python tools/fa_stamps.py
set -e
cd "$(dirname "$0")/../vllm_amd/csrc"
make libvllm_amd_probe.so -j8 > /dev/null
for a in "$@"; do
  build() {   # file, more flags (as in the Makefile)
    /opt/rocm/bin/hipcc --offload-arch=gfx950 -Xclang -target-feature -Xclang -packed-fp32-ops -O3 -std=c++17 -fPIC -fno-gpu-rdc -DNDEBUG -DVA_PROBES -DVA_FA_ABL=$a "${@:2}" -c $1.hip -o build/abl${a}_$1.o
  }
  build prefill_fa
  build prefill_fa_wide -mllvm -amdgpu-mfma-vgpr-form=1
  objs=$(ls build/probe_*.o | grep -v -e 'probe_prefill_fa\.o$' -e 'probe_prefill_fa_wide\.o$' -e 'probe_prefill_fa_abl')
  /opt/rocm/bin/hipcc --offload-arch=gfx950 -shared -fPIC -Wl,-z,defs -o libvllm_amd_probe_abl$a.so $objs build/abl${a}_prefill_fa.o build/abl${a}_prefill_fa_wide.o
done
