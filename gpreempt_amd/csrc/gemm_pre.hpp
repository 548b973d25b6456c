// A per-channel scale, shift and ReLU on the A operand of a matrix product, done where the operand already is: in LDS.
//
// Why: in a network whose normalisation stands in front of its convolutions (DenseNet) every pointwise convolution has a
// scale-shift-ReLU launch in front of it that moves a megabyte and takes 4 us and the 1.4 us between two launches.  The
// bodies that stream their operands through LDS (gemm_pipe.hpp, gemm_wide.hpp) do it themselves, template parameter PRE:
// a wavefront waits for the rows of A that it has fetched, as it does anyway, transforms them in place, 16 bytes per lane and load,
// and the barrier that makes a stage visible makes the transformed rows visible.  In the wide bodies the wavefronts that only
// fetch do it while the first four still multiply the stage before.  Every workgroup of a tile row repeats it, which the vector
// units have time for.  98 of the 309 launches of DenseNet-201 go: batch 4 fp16 1987 -> 1694 us a pass, batch 1 fp32 2690 -> 2458, batch 16
// bf16 2747 -> 2312.
//
// The scale and shift of all K channels lie behind the ring (pre_table_bytes), fetched in front of the first stage.
//
// Same bits as the two launches: the value is rounded to the storage type as it would be on its way through memory, and in
// between computed as the element-wise kernels do, product and sum rounded one by one.  (In fp16 the product of two values is
// exact in fp32, so that one fused multiply-add is the same; the product of two bf16 values can leave fp32's range at either end.)
#pragma once
#include "elementwise_bodies.hpp"

namespace gp {

constexpr size_t kPreMaxTable = 24 * 1024, kPreMaxLds = 159 * 1024;  // the table's bytes, and with the ring (1 KB is left to the dispatcher's and the body's own words)
inline __host__ __device__ constexpr size_t pre_max_lds(size_t ring) { return ring + kPreMaxTable < kPreMaxLds ? ring + kPreMaxTable : kPreMaxLds; }
// scale, then shift, each in whole kilobytes (what one load instruction of a wavefront fetches)
inline __host__ __device__ unsigned pre_table_bytes(int K, unsigned es) { return 2u * (((unsigned)K * es + 1023u) & ~1023u); }

template <typename T> __device__ __forceinline__ out_u32x4 pre_chunk(out_u32x4 x, out_u32x4 scale, out_u32x4 shift, bool relu) {
#pragma clang fp contract(off)  // (product and sum are rounded one by one)
    constexpr int VEC = VecIO<T>::VEC;
    float v[VEC], s[VEC], t[VEC];
    VecIO<T>::unpack(x, v);
    VecIO<T>::unpack(scale, s);
    VecIO<T>::unpack(shift, t);
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
        if constexpr (__is_same(T, _Float16)) v[j] = __builtin_fmaf(v[j], s[j], t[j]);
        else v[j] = v[j] * s[j] + t[j];
    }
    if (relu) {
#pragma unroll
        for (int j = 0; j < VEC; ++j) v[j] = act_f(v[j], GP_ACT_RELU);
    }
    return VecIO<T>::pack(v);
}

}  // namespace gp
