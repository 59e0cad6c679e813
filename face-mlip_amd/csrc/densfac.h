// Factor density of 20 monomials and B = 16 radial functions on split bf16 products (densfac.hip), launched
// by face_density_fwd / face_density_bwd for K a multiple of 16 up to 64.
#pragma once
#include "edges.h"

namespace face {

int launch_density_fwd_limb(const float* phi, int ld_phi, const float* msg, int ld_msg, const int32_t* msg_row,
                            const float* Y, int ld_Y, const int32_t* row_ptr, int64_t N, int M, int K, const RankOut& D,
                            hipStream_t st);
int launch_density_bwd_limb(const float* phi, int ld_phi, const float* msg, int ld_msg, const int32_t* msg_row,
                            const float* Y, int ld_Y, const int32_t* row_ptr, int64_t N, int M, int max_row, int K,
                            const RankIn& G, float* dphi, int ld_dphi, float* dmsg, int ld_dmsg, float* dY, int ld_dY,
                            hipStream_t st);

}  // namespace face
