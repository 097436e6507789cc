// f32 (and f32 x f16) products on bf16 matrix instructions, operands held whole as sums of bf16 parts (ft_split.hip).
#pragma once
#include <cstddef>

struct ft_context;
struct ft_lora_linear_desc;

// out[M, N] = a @ b (+ a2 @ b2) (+ add) for the layouts of the plain products (0: a @ b, 1: a @ b^T, 2: a^T @ b).
bool ft_split_gemm_ok(int layout, size_t M, size_t K, size_t N, bool half_b);
int ft_split_gemm(ft_context* ctx, int layout, bool half_b, const float* a, const void* b, float* out, size_t M,
                  size_t K, size_t N, const float* a2, const float* b2, size_t K2, const float* add);

// y_i = x @ w_i (+ t_i @ b_i) (rotated, or + residual_i) for up to three linears of one input, and gate, up and
// silu(gate) * up of one input: each product as ft_split_gemm_ok says, rotated outputs in whole heads of 64.
int ft_split_group(ft_context* ctx, const float* x, const ft_lora_linear_desc* linears, size_t count, size_t M, size_t K,
                   bool half_b);
int ft_split_gate_up(ft_context* ctx, const float* x, const void* w_gate, const void* w_up, float* gate, float* up,
                     float* act, size_t M, size_t K, size_t N, bool half_b);
