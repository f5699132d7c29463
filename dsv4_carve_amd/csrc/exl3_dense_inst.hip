// Instantiates the dense kernels for one bit width (EXL3_BITS, set by the build).
#include "exl3_dense.hpp"

#ifndef EXL3_BITS
#error "EXL3_BITS must be defined (1..8)"
#endif

namespace exl3 {

template <>
int launch_dequant<EXL3_BITS>(const DequantArgs& a) {
    constexpr int B = EXL3_BITS;
    auto go = [&](auto cbc) {
        constexpr int C = decltype(cbc)::value;
        if (a.suh) {
            const int blocks = (a.k16 / 8) * (a.n16 / 8);
            if (a.nk)
                hipLaunchKernelGGL((dequant_had_kernel<B, C, true>), dim3(blocks), dim3(512), 0, a.stream, a.trellis,
                                   a.k16, a.n16, a.suh, a.svh, a.out);
            else
                hipLaunchKernelGGL((dequant_had_kernel<B, C, false>), dim3(blocks), dim3(512), 0, a.stream,
                                   a.trellis, a.k16, a.n16, a.suh, a.svh, a.out);
        } else {
            const int tiles = a.k16 * a.n16;
            if (a.nk)
                hipLaunchKernelGGL((dequant_raw_kernel<B, C, true>), dim3((tiles + 63) / 64), dim3(64), 0, a.stream,
                                   a.trellis, a.k16, a.n16, a.out);
            else
                hipLaunchKernelGGL((dequant_raw_kernel<B, C, false>), dim3((tiles + 63) / 64), dim3(64), 0,
                                   a.stream, a.trellis, a.k16, a.n16, a.out);
        }
    };
    switch (a.codebook) {
        case CB_MCG: go(std::integral_constant<int, CB_MCG>{}); break;
        case CB_3INST: go(std::integral_constant<int, CB_3INST>{}); break;
        default: go(std::integral_constant<int, CB_MUL1>{}); break;
    }
    return check_launch();
}

// Up to 16 rows: one MFMA row block; 17-32 rows: two.
template <>
int launch_gemv<EXL3_BITS>(const GemvArgs& a) {
    constexpr int B = EXL3_BITS;
    const GemvPlan& p = a.plan;
    const dim3 grid(p.n_hb * p.n_kc), block(WAVE * GEMV_NCG * p.nkg);
    const int lds = gemv_lds_bytes(a.R, p.nsteps, p.nkg);
    auto go = [&](auto cbc) {
        constexpr int C = decltype(cbc)::value;
        auto launch = [&](auto rbc) {
            hipLaunchKernelGGL((gemv_kernel<B, C, decltype(rbc)::value>), grid, block, lds, a.stream, a.x, a.trellis,
                               a.suh, a.svh, a.out, a.out_kind, a.R, a.K, a.N, p.nsteps, p.n_kc, p.xcd ? 1 : 0,
                               a.partials);
        };
        if (a.R > MAX_ROWS) launch(std::integral_constant<int, 2>{});
        else launch(std::integral_constant<int, 1>{});
    };
    switch (a.codebook) {
        case CB_MCG: go(std::integral_constant<int, CB_MCG>{}); break;
        case CB_3INST: go(std::integral_constant<int, CB_3INST>{}); break;
        default: go(std::integral_constant<int, CB_MUL1>{}); break;
    }
    return check_launch();
}

template <>
int launch_gemm<EXL3_BITS>(const GemmArgs& a) {
    constexpr int B = EXL3_BITS;
    const GemmPlan& p = a.plan;
    const dim3 grid(p.n_hb * GEMV_NCG * p.n_kc * p.n_rt), block(WAVE * GEMM_NKG);
    auto go = [&](auto cbc) {
        constexpr int C = decltype(cbc)::value;
        auto launch = [&](auto rbc) {
            constexpr int RB = decltype(rbc)::value;
            constexpr int lds = 4 * RB * (GEMM_NKG - 1) * WAVE * (int)sizeof(float4_t);
            hipLaunchKernelGGL((gemm_kernel<B, C, RB>), grid, block, lds, a.stream, a.xd, a.trellis, p.n_rt * 16 * p.rb,
                               a.K, a.N, p.nsteps, p.n_kc, p.n_rt, a.xcd ? 1 : 0, a.partials);
        };
        switch (p.rb) {
            case 2: launch(std::integral_constant<int, 2>{}); break;
            case 3: launch(std::integral_constant<int, 3>{}); break;
            case 4: launch(std::integral_constant<int, 4>{}); break;
            default: launch(std::integral_constant<int, 5>{}); break;
        }
    };
    switch (a.codebook) {
        case CB_MCG: go(std::integral_constant<int, CB_MCG>{}); break;
        case CB_3INST: go(std::integral_constant<int, CB_3INST>{}); break;
        default: go(std::integral_constant<int, CB_MUL1>{}); break;
    }
    return check_launch();
}

template <>
int launch_gemv_fan<EXL3_BITS>(const FanParams& P, int codebook, hipStream_t stream) {
    constexpr int B = EXL3_BITS;
    const dim3 grid(P.hb0[P.count] * P.n_kc), block(WAVE * GEMV_NCG * P.nkg);
    const int lds = gemv_lds_bytes(P.R, P.nsteps, P.nkg);
    auto go = [&](auto cbc) {
        constexpr int C = decltype(cbc)::value;
        if (P.R > MAX_ROWS) hipLaunchKernelGGL((gemv_fan_kernel<B, C, 2>), grid, block, lds, stream, P);
        else hipLaunchKernelGGL((gemv_fan_kernel<B, C, 1>), grid, block, lds, stream, P);
    };
    switch (codebook) {
        case CB_MCG: go(std::integral_constant<int, CB_MCG>{}); break;
        case CB_3INST: go(std::integral_constant<int, CB_3INST>{}); break;
        default: go(std::integral_constant<int, CB_MUL1>{}); break;
    }
    return check_launch();
}

}  // namespace exl3
