// mrhs.hip -- H-MVM for several right-hand sides on the matrix cores.
//
// Y += a op(A) X with X, Y column-major.  Same plan layout and phases as the
// single right-hand-side path, with the inner products done as 16 x 16 x 4
// MFMA tiles:
//   forward     V pass -> partial sums -> R pass
//   transposed  R pass -> partial sums -> V pass
//               FP64 factors v_mfma_f64_16x16x4f64, the other formats
//               decoded to FP32, v_mfma_f32_16x16x4f32; the transposed V pass
//               FP64 tiles for every format
// Right-hand sides are processed in tiles of 16.
//
//   k_xtrans   XT = X^T, the right-hand sides of an index contiguous
//   k_vfwd_mm  P(c, r) = sum_i V(i, c) X(i, r)      workgroup per V segment
//   k_rtrn_mm  Q(c, r) = sum_i R(i, c) X(i, r)      workgroup per R chunk
//   k_psum_mm  t_e = S_e sum of the entry's partials (FP64 sums)
//   k_ufwd_mm  Y(i, r) += a sum_c R(i, c) Z(c, r)   workgroup per row panel
//   k_vtrn_mm  Y(i, r) += a (sum_c V(i, c) t_c + dense partials)
//                                                   workgroup per column panel

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "kernels.hpp"
#include "mrhs.hpp"
#include "mrhs_dev.hpp"

namespace hmvm {
namespace {

// the wave of the workgroup, as a wave-uniform value
__device__ inline int wave_index() { return __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)); }

template <typename XT, typename WT>
__global__ __launch_bounds__(kThr) void k_xtrans(const XT* __restrict__ X, int64_t ldx, int64_t n, int R,
                                                 WT* __restrict__ XTb) {
    extern __shared__ double tile[];
    xtrans_tile<XT, WT>(X, ldx, n, R, XTb, int64_t(blockIdx.x) * 64, reinterpret_cast<WT*>(tile), threadIdx.x);
}

template <int NTM, typename KIND, typename WT = typename KIND::WT>
__global__ __launch_bounds__(kThr, (mm_reduce_waves<NTM, KIND>())) void k_vfwd_mm(DevPlan P, const WT* __restrict__ XTb,
                                                                              int Rs, WT* __restrict__ Pb) {
    const VItem sg = P.fitems[blockIdx.x];
    vseg_mm<NTM, KIND::FAM, WT>(P, sg, XTb, Rs, Pb, wave_index(), threadIdx.x & 63);
}

template <int NTM, typename KIND, typename WT = typename KIND::WT>
__global__ __launch_bounds__(kThr, (mm_rtrn_waves<NTM, KIND>())) void k_rtrn_mm(DevPlan P, const WT* __restrict__ XTb,
                                                                              int Rs, WT* __restrict__ Q) {
    __shared__ __align__(16) unsigned char tiles[kThr / 64][kTileBytes];
    const RChunk C = P.rchunks[blockIdx.x];
    const int wave = wave_index();
    rchunk_trn_mm<NTM, KIND::FAM, WT>(P, C, XTb, Rs, Q, tiles[wave], wave, threadIdx.x & 63);
}

// one item (entry, NP right-hand sides: a unit of rhs_unit) per thread
template <int NP, typename WT>
__global__ __launch_bounds__(256) void k_psum_mm(DevPlan D, const int32_t* __restrict__ off,
                                                 const int32_t* __restrict__ cnt, const WT* __restrict__ Pb,
                                                 WT* __restrict__ t, int Rs) {
    const int64_t g = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    psum_mm_items<NP, WT, 1, kPsumRound>(D, D.trel, off, cnt, Pb, t, Rs, 1.0, g, 0, D.ntent * (Rs / NP));
}

template <int NW, int NTM, typename YT, typename KIND, typename WT = typename KIND::WT>
__global__ __launch_bounds__(64 * NW, (mm_apply_waves<NTM, KIND>())) void k_ufwd_mm(DevPlan P, double alpha,
                                                                             const WT* __restrict__ z,
                                                                             YT* __restrict__ Y, int64_t ldy, int R) {
    extern __shared__ double red[];
    // runs of 32 consecutive row panels per XCD: the panels of one block row
    // gather the same t and XT rows, which then come from that XCD's L2
    const RowPanel Rw = P.rp[xcd_item(blockIdx.x, P.nrp, 32)];
    rpanel_mm<NW, NTM, YT, KIND::FAM, KIND::k32, WT>(P, Rw, alpha, z, Y, ldy, R, red, threadIdx.x, wave_index(),
                                                 threadIdx.x & 63);
}

template <int NTM, typename YT, typename KIND, typename WT = typename KIND::WT>
__global__ __launch_bounds__(kThr, (mm_vtrn_waves<NTM, KIND>())) void k_vtrn_mm(DevPlan P, double alpha,
                                                                            const WT* __restrict__ z,
                                                                            const WT* __restrict__ Q,
                                                                            YT* __restrict__ Y, int64_t ldy, int R) {
    extern __shared__ double red[];
    const ColPanel C = P.cp[xcd_item(blockIdx.x, P.ncp, 32)];
    cpanel_trn_mm<NTM, YT, KIND::FAM, WT>(P, C, alpha, z, Q, Y, ldy, R, red, threadIdx.x, wave_index(),
                                          threadIdx.x & 63);
}

} // namespace

int launch_apply_mrhs(const DevPlan& D, int fam, bool rows64, bool trans, double alpha, const void* x, int64_t ldx,
                      void* y, int64_t ldy, int R, int vdt, double* ws, hipStream_t st) {
    if (R < 1 || R > kMaxRp) return 1;
    if (fam != kFamHw && fam != kFamBfp && fam != kFamF64 && fam != kFamAfl) return 1;
    const int64_t nin = trans ? D.nrows : D.ncols;
    auto blocks = [](int64_t n, int per) { return unsigned((n + per - 1) / per); };
    auto run = [&](auto kind, auto ntm, auto ytag) {
        using KIND = decltype(kind);
        using WT = typename KIND::WT;
        using YT = decltype(ytag);
        constexpr int NTM = decltype(ntm)::value;
        const int Rs = rhs_stride<WT>(R);
        // workspace, rows of Rs values at 16-byte boundaries: partials | z rows.
        // Forward: t | XT (zero row last).  Transposed: t takes the place of
        // XT, which the sums no longer need; XT lies at its end, so that the
        // zero row stays behind both.
        WT* part = reinterpret_cast<WT*>((reinterpret_cast<uintptr_t>(ws) + 15) & ~uintptr_t(15));
        WT* t = part + (trans ? D.qsize : D.psize) * Rs;
        WT* xt = t + (trans ? trn_zero_row(D) - nin : D.ntent) * Rs;
        YT* Y = static_cast<YT*>(y);
        k_xtrans<YT, WT><<<unsigned(xtrans_tiles(nin)), kThr, xtrans_lds_bytes(R), st>>>(static_cast<const YT*>(x), ldx,
                                                                                         nin, R, xt);
        if (trans) {
            if (D.nrchunks > 0) k_rtrn_mm<NTM, KIND><<<unsigned(D.nrchunks), kThr, 0, st>>>(D, xt, Rs, part);
        } else {
            if (D.nfitems > 0) k_vfwd_mm<NTM, KIND><<<unsigned(D.nfitems), kThr, 0, st>>>(D, xt, Rs, part);
        }
        if (D.ntent > 0) {
            const int32_t* off = trans ? D.qt_off : D.pt_off;
            const int32_t* cnt = trans ? D.qt_cnt : D.pt_cnt;
            auto sums = [&](auto np) {
                constexpr int NP = decltype(np)::value;
                k_psum_mm<NP, WT><<<blocks(D.ntent * (Rs / NP), 256), 256, 0, st>>>(D, off, cnt, part, t, Rs);
            };
            switch (rhs_unit<WT>(R)) {
            case 1: sums(std::integral_constant<int, 1>()); break;
            case 2: sums(std::integral_constant<int, 2>()); break;
            default: sums(std::integral_constant<int, 16 / int(sizeof(WT))>()); break;
            }
        }
        if (trans) {
            if (D.ncp > 0)
                k_vtrn_mm<NTM, YT, KIND><<<unsigned(D.ncp), kThr, mm_red_bytes(kThr / 64), st>>>(D, alpha, t, part, Y, ldy, R);
        } else {
            auto rows = [&](auto nw) {
                constexpr int NW = decltype(nw)::value;
                k_ufwd_mm<NW, NTM, YT, KIND><<<unsigned(D.nrp), 64 * NW, mm_red_bytes(NW), st>>>(D, alpha, t, Y, ldy, R);
            };
            if (D.nrp == 0) return;
            if constexpr (mm_wide<KIND>()) {
                if (D.rsplit) {
                    rows(std::integral_constant<int, kWideWaves>());
                    return;
                }
            }
            rows(std::integral_constant<int, kThr / 64>());
        }
    };
    // accumulators sized for exactly the ceil(R / 16) tiles of this call; one
    // instantiation per kind of plan, which carries only its own formats'
    // decode paths (and registers)
    by_mm_kind(fam, rows64, [&](auto kind) {
        auto with = [&](auto ntm) {
            if (vdt == 0) run(kind, ntm, double(0));
            else run(kind, ntm, float(0));
        };
        switch ((R + 15) / 16) {
        case 1: with(std::integral_constant<int, 1>()); break;
        case 2: with(std::integral_constant<int, 2>()); break;
        case 3: with(std::integral_constant<int, 3>()); break;
        default: with(std::integral_constant<int, 4>()); break;
        }
    });
    return hipGetLastError() == hipSuccess ? 0 : 2;
}

int64_t mrhs_ws_doubles(int fam, bool rows64, bool trans, int64_t partials, int64_t ntent, int64_t nin, int R) {
    const bool f = mm_float_rows(fam, rows64);
    const int64_t Rs = f ? rhs_stride<float>(R) : rhs_stride<double>(R);
    const int64_t rows = (trans ? std::max(ntent, nin) : ntent + nin) + 1;
    // z rows are addressed with 32-bit byte offsets
    if (rows * Rs * (f ? 4 : 8) > int64_t(UINT32_MAX)) return INT64_MAX;
    return (partials + rows) * Rs / (f ? 2 : 1) + 2;
}

} // namespace hmvm
