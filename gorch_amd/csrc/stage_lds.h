// stage_lds.h — operand stages loaded straight to LDS (raw buffer loads to
// LDS, 16 bytes a lane).
//
// A stage row is CH chunks of 16 bytes (CH = 8: 128 bytes, CH = 4: 64). Chunk
// c of row i sits at position c ^ (i & 7), or c ^ ((i >> 1) & 3) in 64-byte
// rows: 16-row fragment reads of 16 bytes a lane are then free of bank
// conflicts.
#pragma once
#include "common.h"

namespace gh {

// Lane l of a load takes row l / CH of its group of 64 / CH rows and the
// chunk that belongs at position l % CH of that row; `chunk` is the same for
// every group, so a lane's offset is a constant plus a scalar (group row,
// step). Everything goes through the checked offset: rows past the resource
// and a step past the last one (kbyte = kOutOfRange) read as zeros, and so do
// chunks past K when `tail` is kOutOfRange for the lane (0 otherwise).
template <int CH>
struct StageLane {
    int chunk, off;
    __device__ __forceinline__ StageLane(int lane, int ld) {
        const int row = lane / CH;
        chunk = (lane % CH) ^ (CH == 8 ? row : ((row >> 1) & 3));
        off = row * ld + 16 * chunk;
    }
    // copies ROWS rows (stride ld bytes) of the step at byte kbyte to LDS
    template <int ROWS, bool KT>
    __device__ __forceinline__ void issue(char* lds, __amdgpu_buffer_rsrc_t rs, int ld, int kbyte, int tail) const {
        constexpr int RPI = 64 / CH;
#pragma unroll
        for (int i = 0; i < ROWS / RPI; i++) {
            unsigned o = (unsigned)off + (unsigned)(i * RPI * ld + kbyte);
            if constexpr (KT) o = max(o, (unsigned)tail);
            typedef __attribute__((address_space(3))) void* lds_ptr;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr)(lds + i * 1024), 16, (int)o, 0, 0, 0);
        }
    }
};

// s_waitcnt operand: vmcnt(VM), lgkmcnt 0 or ignored
constexpr int wait_vm(int vm, bool lgkm0) {
    return (vm & 15) | (7 << 4) | (lgkm0 ? 0 : 15 << 8) | ((vm >> 4) << 14);
}
constexpr int kWaitLgkm0 = 0xc07f;  // lgkmcnt(0) alone

}  // namespace gh
