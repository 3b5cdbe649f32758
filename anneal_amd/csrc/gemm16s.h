// gemm16s.h — f16 contractions whose output has few tiles, or whose sizes are no multiple of a tile (gemm16s.hip).
#pragma once
#include "gemm.h"

namespace ah {

// Launches d on the split kernel and returns true when its operands admit it (the contiguous dimension of each a multiple
// of 8 and 16-byte aligned, under 2 GiB; the store, bias, mask and SGD epilogues without partial sums) and the shape is
// one it serves better than the whole-tile variants (gemm16s.hip has the rule); else returns false.
bool gemm16s_try_launch(const GemmDesc &d, hipStream_t s, hipError_t *err);
bool gemm16s_serves(const GemmDesc &d);

// One tile configuration: split workgroups per tile, each contracting `stages` K stages.
struct G16SPlan {
    int cfg, split, stages;
};
hipError_t gemm16s_launch_0(const GemmDesc &d, const G16SPlan &p, hipStream_t s);
hipError_t gemm16s_launch_1(const GemmDesc &d, const G16SPlan &p, hipStream_t s);
hipError_t gemm16s_launch_2(const GemmDesc &d, const G16SPlan &p, hipStream_t s);
hipError_t gemm16s_launch_3(const GemmDesc &d, const G16SPlan &p, hipStream_t s);
hipError_t gemm16s_launch_4(const GemmDesc &d, const G16SPlan &p, hipStream_t s);
hipError_t gemm16s_launch_5(const GemmDesc &d, const G16SPlan &p, hipStream_t s);
hipError_t gemm16s_launch_6(const GemmDesc &d, const G16SPlan &p, hipStream_t s);
hipError_t gemm16s_launch_7(const GemmDesc &d, const G16SPlan &p, hipStream_t s);
hipError_t gemm16s_launch_8(const GemmDesc &d, const G16SPlan &p, hipStream_t s);

// Tile rows, tile columns and K per stage of each configuration.
struct G16SCfg {
    int bm, bn, bk;
};
constexpr int kG16SConfigs = 9;
constexpr G16SCfg kG16SCfg[kG16SConfigs] = {{128, 128, 64}, {64, 128, 64}, {64, 64, 64}, {32, 64, 128}, {128, 64, 64}, {256, 256, 64}, {128, 128, 64},
                                               {64, 128, 64}, {64, 64, 64}};

}  // namespace ah
