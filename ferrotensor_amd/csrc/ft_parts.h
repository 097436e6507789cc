// f32 values as sums of bf16 numbers: what the product and attention kernels on bf16 parts share (ft_split.hip says what the
// parts hold).
#pragma once
#include <hip/hip_runtime.h>

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

// Two values rounded to bf16, packed as a matrix operand wants them.
__device__ __forceinline__ unsigned pack2(float x, float y) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{x, y}, bf16x2));
}
// The two halves of a packed pair as f32. (v_dot2_f32_bf16 with (-1, 0) would unpack and subtract in one instruction,
// but it runs in the matrix unit: measured, an MFMA and eight of them take as long as both apart, with eight of these
// they take 20 ns where the MFMA alone takes 16.)
__device__ __forceinline__ float low_half(unsigned p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float high_half(unsigned p) { return __uint_as_float(p & 0xffff0000u); }

// What is left of two values before their third part is taken, collected as bits: a third part holds its value when the low
// half of that value is zero (from 2^-110 up, always). (In C the compiler keeps the values and combines them at the end of a
// loop's body, with all the registers that takes.)
__device__ __forceinline__ void collect_left(unsigned& left, float x, float y) {
    asm("v_or3_b32 %0, %0, %1, %2" : "+v"(left) : "v"(x), "v"(y));
}
__device__ __forceinline__ bool left_over(unsigned left) { return (left & 0xffffu) != 0; }
