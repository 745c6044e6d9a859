// Kernel lookup across the separately compiled kernel families (kinst2d.hip,
// kspec2d.hip, kinst1d.hip).  Host-side only.
#pragma once
#include "scat1d_body.h"
#include "scat2d_bwd.h"

template <class T> using Scat2DKernel = void (*)(Scat2DArgs<T>);
template <class T> using Scat1DKernel = void (*)(Scat1DArgs<T>);

Scat2DKernel<float> kym_pick2d_f32_p7(int kind, int threads);
Scat2DKernel<float> kym_pick2d_f32_p17(int kind, int threads);
Scat2DKernel<float> kym_pick2d_f32_p31(int kind, int threads);
Scat2DKernel<float> kym_pick2d_f32_p119(int kind, int threads);
Scat2DKernel<float> kym_pick2d_f32_p123(int kind, int threads);
Scat2DKernel<float> kym_pick2d_f32_p129(int kind, int threads);
Scat2DKernel<float> kym_pick2d_f32_p131(int kind, int threads);
Scat2DKernel<float> kym_pick2d_f32_g7(int kind, int threads);
Scat2DKernel<float> kym_pick2d_f32_g17(int kind, int threads);
Scat2DKernel<float> kym_pick2d_f32_g31(int kind, int threads);
Scat2DKernel<double> kym_pick2d_f64_p7(int kind, int threads);
Scat2DKernel<double> kym_pick2d_f64_p17(int kind, int threads);
Scat2DKernel<double> kym_pick2d_f64_p31(int kind, int threads);
Scat2DKernel<double> kym_pick2d_f64_p119(int kind, int threads);
Scat2DKernel<double> kym_pick2d_f64_p123(int kind, int threads);
Scat2DKernel<double> kym_pick2d_f64_p129(int kind, int threads);
Scat2DKernel<double> kym_pick2d_f64_p131(int kind, int threads);
Scat2DKernel<double> kym_pick2d_f64_g7(int kind, int threads);
Scat2DKernel<double> kym_pick2d_f64_g17(int kind, int threads);
Scat2DKernel<double> kym_pick2d_f64_g31(int kind, int threads);
Scat2DKernel<float> kym_pick_node_spec_f32(int id);
Scat2DKernel<float> kym_pick_bwd_node_spec_f32(int id);
Scat2DKernel<float> kym_pick_pass_spec_f32(int kind, int id);
Scat1DKernel<float> kym_pick1d_f32(int threads, int kind);
Scat1DKernel<float> kym_pick_node1d_spec_f32(int id);
Scat1DKernel<float> kym_pick_bwd_node1d_spec_f32(int id);
Scat1DKernel<float> kym_pick_any1d_f32(int kind);
Scat1DKernel<double> kym_pick1d_f64(int threads, int kind);

// pclass: 7, 17, 31 or 100 + p (kym_plan_class), or KYM_GLOBAL_TW + 7, 17 or 31;
// spec >= 0 selects a compile-time specialisation of the node or pass kernel.
template <class T>
inline Scat2DKernel<T> pick_scat2d(int kind, int threads, int pclass, int spec = -1) {
#define KYM_PICK_FAMILY(tag)                                                  \
    switch (pclass) {                                                         \
        case 7: return kym_pick2d_##tag##_p7(kind, threads);                  \
        case 17: return kym_pick2d_##tag##_p17(kind, threads);                \
        case 119: return kym_pick2d_##tag##_p119(kind, threads);              \
        case 123: return kym_pick2d_##tag##_p123(kind, threads);              \
        case 129: return kym_pick2d_##tag##_p129(kind, threads);              \
        case 131: return kym_pick2d_##tag##_p131(kind, threads);              \
        case KYM_GLOBAL_TW + 7: return kym_pick2d_##tag##_g7(kind, threads);  \
        case KYM_GLOBAL_TW + 17: return kym_pick2d_##tag##_g17(kind, threads); \
        case KYM_GLOBAL_TW + 31: return kym_pick2d_##tag##_g31(kind, threads); \
        default: return kym_pick2d_##tag##_p31(kind, threads);                \
    }
    if constexpr (sizeof(T) == 4) {
        if (spec >= 0 && kind == K2_LDS_NODE) return kym_pick_node_spec_f32(spec);
        if (spec >= 0 && kind == K2B_NODE) return kym_pick_bwd_node_spec_f32(spec);
        if (spec >= 0) return kym_pick_pass_spec_f32(kind, spec);
        KYM_PICK_FAMILY(f32)
    } else {
        KYM_PICK_FAMILY(f64)
    }
#undef KYM_PICK_FAMILY
}

// spec >= 0 (FP32 nodes) selects a compile-time specialisation.
template <class T>
inline Scat1DKernel<T> pick_scat1d(int threads, int kind = 0, int spec = -1) {
    if (spec == KYM_N1_NOSPLIT && kind == 0) kind = 3, spec = -1;
    if constexpr (sizeof(T) == 4) {
        if (spec == KYM_N1_ANY && kind <= 1) return kym_pick_any1d_f32(kind);
        if (spec >= 0 && kind == 0) return kym_pick_node1d_spec_f32(spec);
        if (spec >= 0 && kind == 1) return kym_pick_bwd_node1d_spec_f32(spec);
        return kym_pick1d_f32(threads, kind);
    } else {
        return kym_pick1d_f64(threads, kind);
    }
}
