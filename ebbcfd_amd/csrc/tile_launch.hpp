// Launches of the gradient and tile kernels for one cell stride S.  Each is instantiated in an
// object of its own (gradient.hip, face_tiles.hip, face_batch.hip and grad_tiles.hip, compiled
// once per stride).
#pragma once
#include "dev.hpp"

namespace ebb {

// Epilogue workgroups come first in a launch; the count is padded to whole rounds over the 8
// XCDs, so the workgroups after them keep the XCD the slices of xcdBlock assume.
inline uint32_t epiPadding(uint32_t nEpi) { return (nEpi + 7u) / 8u * 8u; }

template <int S>
void gradS(const DevMesh& m, const PhysParams& p, const StageArgs& a, const DiagArgs& d, hipStream_t st);
template <int S, int MIX>
void gradBatchS(int mode, const MemberArgs* mem, const uint2* items, uint32_t n, uint32_t par, uint32_t st,
                const uint2* epi, uint32_t nEpi, hipStream_t s);
template <int S>
void faceTileS(const DevMesh& m, const PhysParams& p, const StageArgs& a, const FaceTileArgs& t, hipStream_t st);
template <int S>
void gradTileS(const DevMesh& m, const PhysParams& p, const StageArgs& a, const FaceTileArgs& t, int mode, int parts,
               const DiagArgs* epi, hipStream_t st);
template <int S, int MIX>
void faceBatchS(const GroupShape& gs, int limitStage, const MemberArgs* mem, const uint2* items, uint32_t n,
                uint32_t lds, uint32_t par, uint32_t stg, hipStream_t s);
template <int S, int MIX>
void borderBatchS(int mode, const MemberArgs* mem, const uint2* items, uint32_t n, uint32_t par, uint32_t st,
                  const uint2* epi, uint32_t nEpi, hipStream_t s);
template <int S, int MIX>
void gradTileBatchS(const GroupShape& gs, int limitStage, const MemberArgs* mem, const uint2* items, uint32_t n,
                    uint32_t lds, uint32_t par, uint32_t stg, hipStream_t s);

}  // namespace ebb
