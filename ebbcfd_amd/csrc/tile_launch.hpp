// Launches of the tile kernels for one cell stride S.  Each is instantiated in an object of its
// own (face_tiles.hip, face_batch.hip and grad_tiles.hip, compiled once per stride).
#pragma once
#include "dev.hpp"

namespace ebb {

template <int S>
void faceTileS(const DevMesh& m, const PhysParams& p, const StageArgs& a, const FaceTileArgs& t, hipStream_t st);
template <int S>
void gradTileS(const DevMesh& m, const PhysParams& p, const StageArgs& a, const FaceTileArgs& t, int mode, int parts,
               hipStream_t st);
template <int S, int MIX>
void faceBatchS(const GroupShape& gs, int limitStage, const MemberArgs* mem, const uint2* items, uint32_t n,
                uint32_t lds, uint32_t par, uint32_t stg, hipStream_t s);
template <int S, int MIX>
void borderBatchS(int mode, const MemberArgs* mem, const uint2* items, uint32_t n, uint32_t par, uint32_t st,
                  hipStream_t s);
template <int S, int MIX>
void gradTileBatchS(const GroupShape& gs, int limitStage, const MemberArgs* mem, const uint2* items, uint32_t n,
                    uint32_t lds, uint32_t par, uint32_t stg, hipStream_t s);

}  // namespace ebb
