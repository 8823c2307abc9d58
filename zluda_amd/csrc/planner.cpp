// Problem validation, lowering to strides, and kernel selection.  Host code only.
//
// The accepted surface follows the reference's (zluda_blaslt/src/impl.rs:257-305 for the
// attributes, zluda_common/src/lib.rs:575-630 for the type maps) extended by what the quantized
// path needs: scale pointers/modes, pointer modes, FP4/UE8M0 types.
#include "planner.hpp"

#include "kernels/store_window.hpp"

#include <algorithm>
#include <cstdlib>
#include <cstring>

namespace zluda_amd {

static int type_bits(uint32_t t) {
  switch (t) {
  case CUDA_R_32F: case CUDA_R_32I: return 32;
  case CUDA_R_16F: case CUDA_R_16BF: return 16;
  case CUDA_R_8I: case CUDA_R_8F_E4M3: case CUDA_R_8F_E5M2: return 8;
  case CUDA_R_4F_E2M1: return 4;
  default: return 0;
  }
}

static bool is_float_in(uint32_t t) {
  return t == CUDA_R_32F || t == CUDA_R_16F || t == CUDA_R_16BF || t == CUDA_R_8F_E4M3 ||
         t == CUDA_R_8F_E5M2 || t == CUDA_R_4F_E2M1;
}

static uint32_t layout_ok(const zluda_matrix_layout &l) {
  if (l.order != CUBLASLT_ORDER_COL && l.order != CUBLASLT_ORDER_ROW) return CUBLAS_STATUS_NOT_SUPPORTED;
  if (!type_bits(l.type)) return CUBLAS_STATUS_NOT_SUPPORTED;
  if (l.rows == 0 || l.cols == 0) return CUBLAS_STATUS_INVALID_VALUE;
  if (l.rows > 0x7fffffffull || l.cols > 0x7fffffffull) return CUBLAS_STATUS_NOT_SUPPORTED;
  const int64_t lead = l.order == CUBLASLT_ORDER_COL ? (int64_t)l.rows : (int64_t)l.cols;
  if (l.ld < lead) return CUBLAS_STATUS_INVALID_VALUE;
  if (l.batch_count < 1) return CUBLAS_STATUS_INVALID_VALUE;
  return CUBLAS_STATUS_SUCCESS;
}

static int convert_scale_mode(int32_t cuda_mode, const void *ptr, bool dry, int32_t *out) {
  switch (cuda_mode) {
  case CUBLASLT_MATMUL_MATRIX_SCALE_SCALAR_32F: *out = ptr ? SCALE_SCALAR : SCALE_NONE; return 0;
  case CUBLASLT_MATMUL_MATRIX_SCALE_OUTER_VEC_32F: *out = SCALE_OUTER_VEC; return (ptr || dry) ? 0 : 1;
  case CUBLASLT_MATMUL_MATRIX_SCALE_VEC32_UE8M0: *out = SCALE_BLOCK32_UE8M0; return (ptr || dry) ? 0 : 1;
  default: return 2;
  }
}

uint32_t lower_problem(const zluda_gemm_problem *p, bool dry, Lowered *out) {
  if (!p || !out) return CUBLAS_STATUS_INVALID_VALUE;
  const zluda_matmul_desc &op = p->op;
  const zluda_matrix_layout &a = p->a, &b = p->b, &d = p->d;
  const zluda_matrix_layout &c = p->c;
  uint32_t st;
  if ((st = layout_ok(a)) || (st = layout_ok(b)) || (st = layout_ok(c)) || (st = layout_ok(d))) return st;
  if (op.transa > CUBLAS_OP_C || op.transb > CUBLAS_OP_C) return CUBLAS_STATUS_INVALID_VALUE;
  const bool ta = op.transa != CUBLAS_OP_N, tb = op.transb != CUBLAS_OP_N;

  GemmArgs g;
  memset(&g, 0, sizeof(g));
  const uint64_t M = d.rows, N = d.cols, K = ta ? a.rows : a.cols;
  if ((ta ? a.cols : a.rows) != M) return CUBLAS_STATUS_INVALID_VALUE;
  if ((tb ? b.cols : b.rows) != K) return CUBLAS_STATUS_INVALID_VALUE;
  if ((tb ? b.rows : b.cols) != N) return CUBLAS_STATUS_INVALID_VALUE;
  if (c.rows != M || c.cols != N) return CUBLAS_STATUS_INVALID_VALUE;
  g.M = (int32_t)M; g.N = (int32_t)N; g.K = (int32_t)K;

  const bool a_col = a.order == CUBLASLT_ORDER_COL, b_col = b.order == CUBLASLT_ORDER_COL;
  // op(A)(i,k): stored (r,c) = ta ? (k,i) : (i,k)
  if (!ta) { g.a_si = a_col ? 1 : a.ld; g.a_sk = a_col ? a.ld : 1; }
  else     { g.a_sk = a_col ? 1 : a.ld; g.a_si = a_col ? a.ld : 1; }
  // op(B)(k,j): stored (r,c) = tb ? (j,k) : (k,j)
  if (!tb) { g.b_sk = b_col ? 1 : b.ld; g.b_sj = b_col ? b.ld : 1; }
  else     { g.b_sj = b_col ? 1 : b.ld; g.b_sk = b_col ? b.ld : 1; }
  g.c_si = c.order == CUBLASLT_ORDER_COL ? 1 : c.ld; g.c_sj = c.order == CUBLASLT_ORDER_COL ? c.ld : 1;
  g.d_si = d.order == CUBLASLT_ORDER_COL ? 1 : d.ld; g.d_sj = d.order == CUBLASLT_ORDER_COL ? d.ld : 1;

  g.batch = d.batch_count;
  if (a.batch_count != g.batch || b.batch_count != g.batch || c.batch_count != g.batch)
    return CUBLAS_STATUS_INVALID_VALUE;
  g.a_sb = a.batch_stride; g.b_sb = b.batch_stride; g.c_sb = c.batch_stride; g.d_sb = d.batch_stride;
  if (g.batch > 65535) return CUBLAS_STATUS_NOT_SUPPORTED;

  g.a_type = a.type; g.b_type = b.type; g.c_type = c.type; g.d_type = d.type;

  // ---- compute / scale type ------------------------------------------------------------------
  const uint32_t ct = op.compute_type;
  const bool int_path = ct == CUBLAS_COMPUTE_32I || ct == CUBLAS_COMPUTE_32I_PEDANTIC;
  const bool f32_path = ct == CUBLAS_COMPUTE_32F || ct == CUBLAS_COMPUTE_32F_PEDANTIC ||
                        ct == CUBLAS_COMPUTE_32F_FAST_16F || ct == CUBLAS_COMPUTE_32F_FAST_16BF ||
                        ct == CUBLAS_COMPUTE_32F_FAST_TF32;
  if (!int_path && !f32_path) return CUBLAS_STATUS_NOT_SUPPORTED;
  if (int_path) {
    if (a.type != CUDA_R_8I || b.type != CUDA_R_8I) return CUBLAS_STATUS_NOT_SUPPORTED;
    if (op.scale_type == CUDA_R_32I) {
      if (d.type != CUDA_R_32I || c.type != CUDA_R_32I) return CUBLAS_STATUS_NOT_SUPPORTED;
      if (op.epilogue != CUBLASLT_EPILOGUE_DEFAULT) return CUBLAS_STATUS_NOT_SUPPORTED;
      g.int_scale = 1;
    } else if (op.scale_type == CUDA_R_32F) {
      if (!(d.type == CUDA_R_8I || d.type == CUDA_R_32I || d.type == CUDA_R_16BF ||
            d.type == CUDA_R_16F || d.type == CUDA_R_32F))
        return CUBLAS_STATUS_NOT_SUPPORTED;
    } else return CUBLAS_STATUS_NOT_SUPPORTED;
  } else {
    if (!is_float_in(a.type) || !is_float_in(b.type)) return CUBLAS_STATUS_NOT_SUPPORTED;
    if (op.scale_type != CUDA_R_32F) return CUBLAS_STATUS_NOT_SUPPORTED;
    if (!(d.type == CUDA_R_32F || d.type == CUDA_R_16F || d.type == CUDA_R_16BF ||
          d.type == CUDA_R_8F_E4M3 || d.type == CUDA_R_8F_E5M2))
      return CUBLAS_STATUS_NOT_SUPPORTED;
    // 16/32-bit inputs: both operands of one type (as in cuBLASLt); 8/4-bit floats may mix
    if (type_bits(a.type) >= 16 && a.type != b.type) return CUBLAS_STATUS_NOT_SUPPORTED;
    if (type_bits(a.type) != type_bits(b.type)) return CUBLAS_STATUS_NOT_SUPPORTED;
  }
  if (!g.int_scale && (c.type == CUDA_R_4F_E2M1 || d.type == CUDA_R_4F_E2M1)) return CUBLAS_STATUS_NOT_SUPPORTED;

  // FP4 is packed two per byte along K
  if (a.type == CUDA_R_4F_E2M1 && (g.a_sk != 1 || (a.ld & 1) || (a.batch_stride & 1))) return CUBLAS_STATUS_NOT_SUPPORTED;
  if (b.type == CUDA_R_4F_E2M1 && (g.b_sk != 1 || (b.ld & 1) || (b.batch_stride & 1))) return CUBLAS_STATUS_NOT_SUPPORTED;
  if ((a.type == CUDA_R_4F_E2M1 || b.type == CUDA_R_4F_E2M1) && (K & 1)) return CUBLAS_STATUS_INVALID_VALUE;

  // ---- alpha / beta ------------------------------------------------------------------------
  switch (op.pointer_mode) {
  case CUBLASLT_POINTER_MODE_HOST: g.alpha_mode = SCALAR_VALUE; g.beta_mode = SCALAR_VALUE; break;
  case CUBLASLT_POINTER_MODE_DEVICE: g.alpha_mode = SCALAR_DEV; g.beta_mode = SCALAR_DEV; break;
  case CUBLASLT_POINTER_MODE_DEVICE_VECTOR: g.alpha_mode = VECTOR_DEV; g.beta_mode = VECTOR_DEV; break;
  case CUBLASLT_POINTER_MODE_ALPHA_DEVICE_VECTOR_BETA_ZERO: g.alpha_mode = VECTOR_DEV; g.beta_mode = SCALAR_VALUE; break;
  case CUBLASLT_POINTER_MODE_ALPHA_DEVICE_VECTOR_BETA_HOST: g.alpha_mode = VECTOR_DEV; g.beta_mode = SCALAR_VALUE; break;
  default: return CUBLAS_STATUS_INVALID_VALUE;
  }
  g.alpha_sb = op.alpha_vector_batch_stride;
  if (op.pointer_mode == CUBLASLT_POINTER_MODE_ALPHA_DEVICE_VECTOR_BETA_ZERO && g.alpha_sb != 0)
    return CUBLAS_STATUS_INVALID_VALUE;  // cuda_types/src/cublaslt.rs:4240-4247
  bool beta_maybe_nonzero = true;
  if (!dry) {
    if (!p->alpha) return CUBLAS_STATUS_INVALID_VALUE;
    if (g.alpha_mode == SCALAR_VALUE) memcpy(&g.alpha_val, p->alpha, 4);
    else g.alpha_ptr = p->alpha;
    if (op.pointer_mode == CUBLASLT_POINTER_MODE_ALPHA_DEVICE_VECTOR_BETA_ZERO) {
      g.beta_val.i = 0;
    } else {
      if (!p->beta) return CUBLAS_STATUS_INVALID_VALUE;
      if (g.beta_mode == SCALAR_VALUE) memcpy(&g.beta_val, p->beta, 4);
      else g.beta_ptr = p->beta;
    }
    if (g.beta_mode == SCALAR_VALUE) beta_maybe_nonzero = g.int_scale ? g.beta_val.i != 0 : g.beta_val.f != 0.0f;
    if (beta_maybe_nonzero && !p->C) return CUBLAS_STATUS_INVALID_VALUE;
    if (!p->A || !p->B || !p->D) return CUBLAS_STATUS_INVALID_VALUE;
  }
  g.A = p->A; g.B = p->B; g.C = p->C; g.D = p->D;

  // ---- scales --------------------------------------------------------------------------------
  int r;
  if ((r = convert_scale_mode(op.a_scale_mode, op.a_scale, dry, &g.a_scale_mode)))
    return r == 1 ? CUBLAS_STATUS_INVALID_VALUE : CUBLAS_STATUS_NOT_SUPPORTED;
  if ((r = convert_scale_mode(op.b_scale_mode, op.b_scale, dry, &g.b_scale_mode)))
    return r == 1 ? CUBLAS_STATUS_INVALID_VALUE : CUBLAS_STATUS_NOT_SUPPORTED;
  if (op.c_scale_mode != CUBLASLT_MATMUL_MATRIX_SCALE_SCALAR_32F ||
      op.d_scale_mode != CUBLASLT_MATMUL_MATRIX_SCALE_SCALAR_32F)
    return CUBLAS_STATUS_NOT_SUPPORTED;
  g.a_scale = op.a_scale; g.b_scale = op.b_scale; g.c_scale = op.c_scale; g.d_scale = op.d_scale;
  if (g.int_scale && (g.a_scale_mode || g.b_scale_mode || g.c_scale || g.d_scale))
    return CUBLAS_STATUS_INVALID_VALUE;  // cuda_types/src/cublaslt.rs:4266-4267
  if (g.a_scale_mode == SCALE_BLOCK32_UE8M0 && (int_path || g.a_sk != 1 || (K % 32))) return CUBLAS_STATUS_NOT_SUPPORTED;
  if (g.b_scale_mode == SCALE_BLOCK32_UE8M0 && (int_path || g.b_sk != 1 || (K % 32))) return CUBLAS_STATUS_NOT_SUPPORTED;

  // ---- epilogue ------------------------------------------------------------------------------
  bool has_bias = false;
  switch (op.epilogue) {
  case CUBLASLT_EPILOGUE_DEFAULT: g.act = ACT_NONE; break;
  case CUBLASLT_EPILOGUE_RELU: g.act = ACT_RELU; break;
  case CUBLASLT_EPILOGUE_GELU: g.act = ACT_GELU; break;
  case CUBLASLT_EPILOGUE_BIAS: g.act = ACT_NONE; has_bias = true; break;
  case CUBLASLT_EPILOGUE_RELU_BIAS: g.act = ACT_RELU; has_bias = true; break;
  case CUBLASLT_EPILOGUE_GELU_BIAS: g.act = ACT_GELU; has_bias = true; break;
  // the bias buffer is an output here: sums over K of op(A)'s rows / op(B)'s columns, D as with DEFAULT
  case CUBLASLT_EPILOGUE_BGRADA: g.act = ACT_NONE; g.bgrad_src = 1; break;
  case CUBLASLT_EPILOGUE_BGRADB: g.act = ACT_NONE; g.bgrad_src = 2; break;
  // GELU with its input kept, and GELU's gradient: in the GEMM kernel's epilogue where aux_in_epilogue() says so; elsewhere it runs
  // without the activation, and a second element-wise pass (kernels/aux_epilogue.hpp) finishes D
  case CUBLASLT_EPILOGUE_GELU_AUX: g.act = ACT_NONE; g.aux_mode = 1; break;
  case CUBLASLT_EPILOGUE_GELU_AUX_BIAS: g.act = ACT_NONE; g.aux_mode = 1; has_bias = true; break;
  case CUBLASLT_EPILOGUE_DGELU: g.act = ACT_NONE; g.aux_mode = 2; break;
  case CUBLASLT_EPILOGUE_DGELU_BGRAD: g.act = ACT_NONE; g.aux_mode = 2; g.aux_bgrad = 1; break;
  default: return CUBLAS_STATUS_NOT_SUPPORTED;
  }
  if (g.aux_mode) {
    // the aux matrix has D's type, shape and order (cuda_types/src/cublaslt.rs:4207-4236: its leading dimension
    // is no less than D's rows); both passes go through D's type, which has to be a float type of 16 or 32 bits
    if (g.int_scale || !(d.type == CUDA_R_32F || d.type == CUDA_R_16F || d.type == CUDA_R_16BF)) return CUBLAS_STATUS_NOT_SUPPORTED;
    if (op.epilogue_aux_type != -1 && (uint32_t)op.epilogue_aux_type != d.type) return CUBLAS_STATUS_NOT_SUPPORTED;
    const int64_t lead = d.order == CUBLASLT_ORDER_COL ? M : N, other = d.order == CUBLASLT_ORDER_COL ? N : M;
    if (op.epilogue_aux_ld < lead) return CUBLAS_STATUS_INVALID_VALUE;
    if (g.batch > 1 && op.epilogue_aux_batch_stride < op.epilogue_aux_ld * other && op.epilogue_aux_batch_stride != 0)
      return CUBLAS_STATUS_INVALID_VALUE;
    if (g.batch > 1 && op.epilogue_aux_batch_stride == 0 && g.aux_mode == 1) return CUBLAS_STATUS_NOT_SUPPORTED;  // aliased outputs
    if (g.aux_mode == 2 && g.d_scale) return CUBLAS_STATUS_NOT_SUPPORTED;  // (the scale would have to follow the gradient)
    if (!dry && !op.epilogue_aux) return CUBLAS_STATUS_INVALID_VALUE;
    g.aux = op.epilogue_aux;
    g.aux_si = d.order == CUBLASLT_ORDER_COL ? 1 : op.epilogue_aux_ld;
    g.aux_sj = d.order == CUBLASLT_ORDER_COL ? op.epilogue_aux_ld : 1;
    g.aux_sb = op.epilogue_aux_batch_stride;
    if (g.aux_bgrad) {
      if (g.batch > 1 && op.bias_batch_stride == 0) return CUBLAS_STATUS_NOT_SUPPORTED;
      if (!dry && !op.bias) return CUBLAS_STATUS_INVALID_VALUE;
      g.bgrad = const_cast<void *>(op.bias);
    }
  }
  if (g.bgrad_src) {
    // sums of the stored elements: defined here for unscaled operands only
    if (a.type == CUDA_R_4F_E2M1 || b.type == CUDA_R_4F_E2M1 || g.a_scale_mode || g.b_scale_mode)
      return CUBLAS_STATUS_NOT_SUPPORTED;
    // batches with no stride between their gradient vectors would all write the same one
    if (g.batch > 1 && op.bias_batch_stride == 0) return CUBLAS_STATUS_NOT_SUPPORTED;
    if (!dry && !op.bias) return CUBLAS_STATUS_INVALID_VALUE;
    g.bgrad = const_cast<void *>(op.bias);
  }
  if (has_bias || g.bgrad_src || g.aux_bgrad) {
    if (has_bias && !dry && !op.bias) return CUBLAS_STATUS_INVALID_VALUE;
    if (has_bias) g.bias = op.bias;
    g.bias_sb = op.bias_batch_stride;
    if (op.bias_type >= 0) g.bias_type = (uint32_t)op.bias_type;
    else  // cuda_types/src/cublaslt.rs:4395-4403
      g.bias_type = (d.type == CUDA_R_8I || d.type == CUDA_R_32I || d.type == CUDA_R_8F_E4M3 ||
                     d.type == CUDA_R_8F_E5M2) ? CUDA_R_32F : d.type;
    if (!(g.bias_type == CUDA_R_32F || g.bias_type == CUDA_R_16F || g.bias_type == CUDA_R_16BF))
      return CUBLAS_STATUS_NOT_SUPPORTED;
  }

  out->g = g;
  out->has_bias = has_bias;
  out->a_kcontig = g.a_sk == 1;
  out->b_kcontig = g.b_sk == 1;
  auto al16 = [](const void *ptr, int64_t pitch_elems, int64_t bstride, int bits, bool batched) {
    return (((uintptr_t)ptr) & 15) == 0 && ((pitch_elems * bits / 8) & 15) == 0 &&
           (!batched || ((bstride * bits / 8) & 15) == 0);
  };
  out->aligned16 = al16(g.A, g.a_si, g.a_sb, type_bits(a.type), g.batch > 1) &&
                   al16(g.B, g.b_sj, g.b_sb, type_bits(b.type), g.batch > 1) &&
                   (((int64_t)K * type_bits(a.type) / 8) & 15) == 0;
  // the MFMA kernels address each operand through a 2 GiB buffer window
  const int64_t span_a = ((int64_t)(M - 1) * g.a_si + (int64_t)K) * type_bits(a.type) / 8;
  const int64_t span_b = ((int64_t)(N - 1) * g.b_sj + (int64_t)K) * type_bits(b.type) / 8;
  out->span_ok = span_a < 0x7fffffffll && span_b < 0x7fffffffll;
  return CUBLAS_STATUS_SUCCESS;
}

static bool is_f8(uint32_t t) { return t == CUDA_R_8F_E4M3 || t == CUDA_R_8F_E5M2; }

static bool decode_variant_ok(const Lowered &l, int variant) {
  const GemmArgs &g = l.g;
  const DecodeVariant &v = kDecodeVariants[variant];
  const int T = std::min(g.M, g.N), nb = (T + 15) / 16;
  const bool h16 = g.a_type == CUDA_R_16F || g.a_type == CUDA_R_16BF;
  const bool mx = g.a_type == CUDA_R_4F_E2M1;
  if ((h16 || mx) && v.stream != 2) return false;  // 16- and 4-bit weights: the slab form only
  // the register-streaming kernel is int8 only; token blocks multiply its fragment registers
  if (!v.stream) return g.a_type == CUDA_R_8I && (nb == 1 || (nb == 2 && v.steps <= 8));
  const bool swapped = g.M < g.N;
  const int64_t rows = swapped ? g.N : g.M, ldw = swapped ? g.b_sj : g.a_si;
  if (v.stream == 2) {
    const int64_t ldx = swapped ? g.a_si : g.b_sj;
    // (the 4-wave shape serves K down to half of its 4096; an 8-wave shape the K above the next smaller cover)
    const int cover = v.nw * v.steps * 64, below = cover == 4096 ? cover / 2 : cover - 4096;
    // one block of tokens; two in the 8-wave shapes of one or two units (the one-unit shape exists for them alone)
    // (MXFP4, whose scales take registers too, has neither two units with two blocks nor four units)
    const bool tokens_ok = v.nw == 4 ? nb == 1 : v.steps == 8 ? nb == 2 : v.steps == 16 ? nb <= (mx ? 1 : 2) : nb == 1 && !(mx && v.steps == 32);
    const int64_t bits = type_bits(g.a_type), kb = (int64_t)g.K * bits / 8;  // covers are bytes of K
    return tokens_ok && kb <= cover && kb > below && (kb & (mx ? 127 : 15)) == 0 && rows * ldw * bits / 8 < 0x7fffffffll &&
           ((int64_t)(T - 1) * ldx + g.K) * bits / 8 < 0x7fffffffll;
  }
  // a stream instantiation covers nw * steps * 64 bytes of K and takes any K up to that (lanes past the end read
  // zero); more than a quarter of idle lanes is left to the smaller instantiations or to the MFMA tiles
  const int cover = v.nw * v.steps * 64;
  return g.K <= cover && g.K * 4 > cover * 3 && (g.K & 15) == 0 && rows * ldw < 0x7fffffffll &&
         nb * v.steps <= kDecodeStreamMaxFragments;
}

static bool any_decode_variant_ok(const Lowered &l) {
  for (int v = 0; v < kNumDecodeVariants; v++)
    if (decode_variant_ok(l, v)) return true;
  return false;
}

static bool d_type_fast(const GemmArgs &g) {
  return g.d_type == CUDA_R_32I || g.d_type == CUDA_R_32F || g.d_type == CUDA_R_16BF || g.d_type == CUDA_R_16F || g.d_type == CUDA_R_8I;
}

// The family of the transposing kernel that runs the operands (TR8: 8-bit, TR16: 16-bit, TR32: f32), each with unit stride
// along K or along its row index, or 0.  The families themselves take dword-aligned operands whose K-contiguous rows are
// whole 16-byte pieces; the kernel takes more (`any_pitch`): 16-bit and f32 operands at any element's address and any
// pitch, and K-contiguous rows that end anywhere.
static uint32_t transposing_family(const Lowered &l, bool any_pitch) {
  const GemmArgs &g = l.g;
  const bool h16 = g.a_type == CUDA_R_16F || g.a_type == CUDA_R_16BF, f32 = g.a_type == CUDA_R_32F;
  const bool i8 = g.a_type == CUDA_R_8I && g.b_type == CUDA_R_8I;
  const bool f8 = is_f8(g.a_type) && is_f8(g.b_type) && !(g.a_type == CUDA_R_8F_E5M2 && g.b_type == CUDA_R_8F_E5M2);
  if (!d_type_fast(g) || g.a_scale_mode == SCALE_BLOCK32_UE8M0 || g.b_scale_mode == SCALE_BLOCK32_UE8M0) return 0;
  if (!(i8 || f8 || ((h16 || f32) && g.b_type == g.a_type))) return 0;
  const int64_t esz = f32 ? 4 : h16 ? 2 : 1;
  const int64_t align = (any_pitch && h16 ? 2 : 4) - 1;
  // (strides in bytes from here on)
  auto operand_ok = [&](const void *ptr, int64_t s_row, int64_t s_k, int64_t s_b, int rows) {
    s_row *= esz; s_k *= esz; s_b *= esz;
    if ((((uintptr_t)ptr) & align) || (g.batch > 1 && (s_b & align))) return false;
    const int64_t span = (int64_t)(rows - 1) * s_row + (int64_t)(g.K - 1) * s_k + esz;
    if (span >= 0x7fffffffll) return false;
    if (s_k == esz) return (s_row & align) == 0 && (any_pitch || ((g.K * esz) & 15) == 0);
    // (offsets of K rows up to three stages past the end must stay below 2^32, where they are out
    // of range instead of wrapping into it)
    return s_row == esz && (s_k & align) == 0 && (int64_t)(g.K + 256) * s_k < 0xffffffffll;
  };
  if (!operand_ok(g.A, g.a_si, g.a_sk, g.a_sb, g.M) || !operand_ok(g.B, g.b_sj, g.b_sk, g.b_sb, g.N)) return 0;
  return f32 ? ZLUDA_KERNEL_MFMA_TR32 : h16 ? ZLUDA_KERNEL_MFMA_TR16 : ZLUDA_KERNEL_MFMA_TR8;
}

bool lds_transposable(const Lowered &l) {
  const GemmArgs &g = l.g;
  if ((g.a_type != CUDA_R_16F && g.a_type != CUDA_R_16BF) || g.b_type != g.a_type || (l.a_kcontig && l.b_kcontig)) return false;
  auto ok = [&](const void *ptr, int64_t s_row, int64_t s_k, int64_t s_b) {
    if ((((uintptr_t)ptr) & 15) || (g.batch > 1 && ((s_b * 2) & 15))) return false;
    if (s_k == 1) return ((s_row * 2) & 15) == 0 && (g.K & 7) == 0;
    // (the K rows of the last stage past the end stay below 2 GiB too: the scalar offset of its loads counts them)
    return s_row == 1 && ((s_k * 2) & 15) == 0 && ((int64_t)g.K + 64) * s_k * 2 < 0x7fffffffll;
  };
  return ok(g.A, g.a_si, g.a_sk, g.a_sb) && ok(g.B, g.b_sj, g.b_sk, g.b_sb);
}

bool family_supports(uint32_t kernel, const Lowered &l) {
  const GemmArgs &g = l.g;
  const bool fast_layout = l.a_kcontig && l.b_kcontig && l.aligned16;
  const bool d_fast = d_type_fast(g);
  switch (kernel) {
  case ZLUDA_KERNEL_GENERIC: return true;
  case ZLUDA_KERNEL_MFMA_I8:
    return fast_layout && l.span_ok && g.a_type == CUDA_R_8I && g.b_type == CUDA_R_8I && d_fast;
  case ZLUDA_KERNEL_MFMA_F8:
    return fast_layout && l.span_ok && is_f8(g.a_type) && is_f8(g.b_type) &&
           !(g.a_type == CUDA_R_8F_E5M2 && g.b_type == CUDA_R_8F_E5M2) &&
           g.a_scale_mode != SCALE_BLOCK32_UE8M0 && g.b_scale_mode != SCALE_BLOCK32_UE8M0 && d_fast;
  case ZLUDA_KERNEL_MFMA_MXF4:
    return fast_layout && l.span_ok && g.a_type == CUDA_R_4F_E2M1 && g.b_type == CUDA_R_4F_E2M1 &&
           g.a_scale_mode == SCALE_BLOCK32_UE8M0 && g.b_scale_mode == SCALE_BLOCK32_UE8M0 &&
           (g.K % 256) == 0 && ((((uintptr_t)g.a_scale) | ((uintptr_t)g.b_scale)) & 3) == 0 && d_fast;
  case ZLUDA_KERNEL_MFMA_H16:
    // f16 x f16 or bf16 x bf16 (lower_problem admits 16-bit operands of one type only)
    return fast_layout && l.span_ok && (g.a_type == CUDA_R_16F || g.a_type == CUDA_R_16BF) && g.b_type == g.a_type &&
           g.a_scale_mode != SCALE_BLOCK32_UE8M0 && g.b_scale_mode != SCALE_BLOCK32_UE8M0 && d_fast;
  case ZLUDA_KERNEL_MFMA_F32:
    return fast_layout && l.span_ok && g.a_type == CUDA_R_32F && g.b_type == CUDA_R_32F && d_fast;
  case ZLUDA_KERNEL_MFMA_TR8: case ZLUDA_KERNEL_MFMA_TR16: case ZLUDA_KERNEL_MFMA_TR32:
    return transposing_family(l, false) == kernel;
  case ZLUDA_KERNEL_DECODE_W8A8:
    // int8, or e4m3 x e4m3 without block scales (the LDS-streaming variants only), or f16 / bf16 or MXFP4 (the slab form only)
    return fast_layout && ((g.a_type == CUDA_R_8I && g.b_type == CUDA_R_8I) ||
                           ((g.a_type == CUDA_R_16F || g.a_type == CUDA_R_16BF) && g.b_type == g.a_type) ||
                           (g.a_type == CUDA_R_4F_E2M1 && family_supports(ZLUDA_KERNEL_MFMA_MXF4, l)) ||
                           (g.a_type == CUDA_R_8F_E4M3 && g.b_type == CUDA_R_8F_E4M3 &&
                            g.a_scale_mode != SCALE_BLOCK32_UE8M0 && g.b_scale_mode != SCALE_BLOCK32_UE8M0)) &&
           std::min(g.M, g.N) <= kDecodeMaxTokens && std::max(g.M, g.N) >= 64 && any_decode_variant_ok(l);
  default: return false;
  }
}

static uint32_t ceil_div(uint32_t a, uint32_t b) { return (a + b - 1) / b; }

int w4_epilogue_class(const Lowered &l, bool dry) {
  const GemmArgs &g = l.g;
  // (GELU with its input kept has an epilogue of its own where a plain problem has W4_CLASS_BF16 and aux_in_epilogue() holds; the other
  // epilogues with an aux matrix are plain problems here: launch_planned points D at the aux matrix or runs the gradient pass behind it)
  if (g.beta_mode != SCALAR_VALUE) return W4_CLASS_NONE;
  const bool swapped = g.d_si != 1;
  const int64_t d_sq = swapped ? g.d_si : g.d_sj;
  const int dbytes = (g.d_type == CUDA_R_32I || g.d_type == CUDA_R_32F) ? 4 : 2;
  if (((d_sq * dbytes) & 15) || (g.batch > 1 && ((g.d_sb * dbytes) & 15)) || d_sq >= kNarrowPitch || (((uintptr_t)g.D) & 15))
    return W4_CLASS_NONE;
  const bool i8 = g.a_type == CUDA_R_8I && g.b_type == CUDA_R_8I;
  if (i8 && g.int_scale) {
    if (g.d_type != CUDA_R_32I || g.alpha_mode == VECTOR_DEV || (!dry && g.beta_val.i != 0)) return W4_CLASS_NONE;
    return W4_CLASS_I32;
  }
  // float epilogues: int8 with float scaling (W8A8: alpha[] or outer scales per row and per token), fp8, f16 and bf16
  const bool h16 = (g.a_type == CUDA_R_16F || g.a_type == CUDA_R_16BF) && g.b_type == g.a_type;
  const bool f8a = g.a_type == CUDA_R_8F_E4M3 || g.a_type == CUDA_R_8F_E5M2, f8b = g.b_type == CUDA_R_8F_E4M3 || g.b_type == CUDA_R_8F_E5M2;
  const bool f8 = f8a && f8b && !(g.a_type == CUDA_R_8F_E5M2 && g.b_type == CUDA_R_8F_E5M2);  // (E5M2 x E5M2 is not a cuBLASLt combination)
  if ((i8 || h16 || f8) && g.a_scale_mode != SCALE_BLOCK32_UE8M0 &&
      g.b_scale_mode != SCALE_BLOCK32_UE8M0) {
    if ((g.d_type != CUDA_R_16BF && g.d_type != CUDA_R_16F && g.d_type != CUDA_R_32F) || (!dry && g.beta_val.f != 0.0f))
      return W4_CLASS_NONE;  // (ReLU and the output type are run-time choices of the two classes)
    // scale vectors may run either way; a bias only along D's unit stride
    if (swapped && l.has_bias) return W4_CLASS_NONE;
    return g.act == ACT_GELU ? W4_CLASS_BF16_GELU : W4_CLASS_BF16;
  }
  if (g.a_type == CUDA_R_4F_E2M1 && g.b_type == CUDA_R_4F_E2M1 && g.a_scale_mode == SCALE_BLOCK32_UE8M0 &&
      g.b_scale_mode == SCALE_BLOCK32_UE8M0) {
    // MXFP4: whole scale chunks (1024 elements of K) per tile, and no vector along D's unit stride either (the scale
    // chunks take the LDS the other kinds stage such vectors in)
    if ((g.d_type != CUDA_R_16BF && g.d_type != CUDA_R_16F && g.d_type != CUDA_R_32F) || (!dry && g.beta_val.f != 0.0f))
      return W4_CLASS_NONE;  // (ReLU and the output type are run-time choices of the two classes)
    if ((g.K & 1023) || g.alpha_mode == VECTOR_DEV || l.has_bias) return W4_CLASS_NONE;
    return g.act == ACT_GELU ? W4_CLASS_BF16_GELU : W4_CLASS_BF16;
  }
  return W4_CLASS_NONE;
}

bool mfma_short_k_operands(const Lowered &l) {
  const GemmArgs &g = l.g;
  if ((g.a_type != CUDA_R_16F && g.a_type != CUDA_R_16BF) || g.K > 128 || std::min(g.M, g.N) <= 64 || g.beta_mode != SCALAR_VALUE) return false;
  if (g.d_type != CUDA_R_16F && g.d_type != CUDA_R_16BF && g.d_type != CUDA_R_32F) return false;
  // (its epilogue has one factor for all of D)
  return g.act == ACT_NONE && !l.has_bias && g.alpha_mode != VECTOR_DEV && g.a_scale_mode != SCALE_OUTER_VEC && g.b_scale_mode != SCALE_OUTER_VEC;
}

// (Columns of D at odd 16-bit addresses are left to the tile kernels, whose narrower stores mind them less: bf16 2459 x 351 x 80, 21
// batches 23.3 us here, 19.4 there; with a pitch of 2462 or 2464 16 here and 18.5 there.)
bool mfma_short_k_output(const Lowered &l, bool dry) {
  const GemmArgs &g = l.g;
  // (the kernel's output: where the GELU input is kept, that matrix)
  const bool aux = g.aux_mode == 1, swapped = g.d_si != 1;
  const int64_t d_sq = aux ? (swapped ? g.aux_si : g.aux_sj) : swapped ? g.d_si : g.d_sj, d_sb = aux ? g.aux_sb : g.d_sb;
  if (d_sq >= kNarrowPitch || (!dry && g.beta_val.f != 0.0f)) return false;
  return g.d_type == CUDA_R_32F || !((d_sq & 1) || (g.batch > 1 && (d_sb & 1)) || (!dry && (((uintptr_t)g.D) & 3)));
}

// All of K in LDS at once and more tiles than the two workgroups of every CU take in one go: those walk the tiles.
static uint32_t short_k_groups(uint32_t cus) { return std::max(2 * cus / 8 * 8, 8u); }
static bool mfma_short_k(const Lowered &l, uint32_t cus) {
  return mfma_short_k_operands(l) && mfma_short_k_output(l, true) &&
         (uint64_t)ceil_div(l.g.M, 128) * ceil_div(l.g.N, 128) * l.g.batch > std::max(2 * cus, short_k_groups(cus));
}

// The 256 x 128 tile has a second form on eight waves with three stages, faster on grids of less than two rounds (int8, us:
// 6144 x 777 x 4096 39.6 -> 30.6, 4096 x 2048 x 4096 42 -> 38, 28672 x 777 x 4096, three rounds, 163 -> 131, where the larger
// tiles take 105).  Results of 4 bytes on a grid that fills the chip need a longer K for it: int8 -> int32 5372 x 1428 x 1536 20.9 us on
// four waves, 24.3 on eight, x 4096 43 and 37; 2048 x 2048 x 1024 13.7 and 12.3.  MXFP4 has no room in LDS for the third stage beside
// its scale chunks.
static bool mfma_eight_waves(const Lowered &l, uint64_t tiles, uint32_t cus) {
  if (l.g.a_type == CUDA_R_4F_E2M1 || tiles >= 2 * (uint64_t)cus) return false;
  const bool wide_d = l.g.d_type == CUDA_R_32I || l.g.d_type == CUDA_R_32F;
  return !wide_d || tiles * 4 <= 3 * (uint64_t)cus || (int64_t)l.g.K * type_bits(l.g.a_type) / 8 > 2048;
}

// Workgroups of a variant that a CU holds: data stages, plus two chunks of 32 scale bytes per tile row for MXFP4
static uint32_t mfma_per_cu(const Lowered &l, const MfmaVariant &v) {
  const uint32_t lds = (uint32_t)v.stages * (v.bp + v.bq) * v.bkb + (l.g.a_type == CUDA_R_4F_E2M1 ? 64u * (v.bp + v.bq) : 0u);
  return std::max(1u, std::min(160u * 1024u / lds, 2048u / (v.wp * v.wq * 64u)));
}

// Split-K: when even the chosen tiles leave half of the CUs idle and K is long, grid_z workgroups
// share a tile's K range, write their fp32 / int32 partial tiles to the workspace and a second
// kernel sums them and applies the epilogue.  Only if the caller's workspace holds the partial
// tiles (padded to whole tiles).  (MXFP4 shares are whole scale chunks: the launcher rounds.)
static uint32_t mfma_splits(const Lowered &l, const MfmaVariant &v, uint64_t tiles, uint32_t cus, uint64_t workspace_size) {
  const GemmArgs &g = l.g;
  if (tiles * 2 > cus) return 1;
  // (below ~6 KiB of K per row the second kernel and the workspace traffic cost more than the idle CUs)
  const uint32_t kbytes = ceil_div((uint32_t)((int64_t)g.K * type_bits(g.a_type) / 8), v.bkb) * v.bkb;
  // Skinny problems (<= 64 rows or columns) are memory bound: they split from 2 KiB of K per row on
  // and down to 1 KiB per share, up to two workgroups per CU (fp8 4096x48x4096: 18 -> 13 us; but
  // 14336x64x4096, 224 tiles, must stay whole: 16.5 us against 23.7 split in three).
  const bool skinny = std::min(g.M, g.N) <= 64;
  const bool mx = g.a_type == CUDA_R_4F_E2M1;  // (a byte of FP4 is worth two K steps: 4096x16x4096 loses when split)
  const uint32_t np = g.d_si != 1 ? g.N : g.M;
  if (kbytes < (skinny ? (mx ? 4096u : 2048u) : 6144u) || (uint64_t)ceil_div(np, v.bp) * v.bp > (1u << 20)) return 1;
  uint32_t s = (uint32_t)std::min<uint64_t>({8, (skinny ? 2 * cus : cus) / tiles, kbytes / (skinny ? 1024 : 2048)});
  while (s > 1 && s * tiles * v.bp * v.bq * 4 > workspace_size) s--;
  return std::max(s, 1u);
}

static void fill_mfma_plan(const Lowered &l, int variant, uint32_t cus, uint64_t workspace_size,
                           zluda_gemm_plan *plan) {
  const GemmArgs &g = l.g;
  const MfmaVariant &v = kMfmaVariants[variant];
  const bool swapped = g.d_si != 1;  // row-major D: compute D^T
  const uint32_t np = swapped ? g.N : g.M, nq = swapped ? g.M : g.N;
  const uint32_t tp = ceil_div(np, v.bp), tq = ceil_div(nq, v.bq);
  plan->variant = variant;
  plan->swapped = swapped;
  plan->grid_x = tp * tq; plan->grid_y = g.batch; plan->grid_z = 1;
  plan->block = v.wp * v.wq * 64;
  if (v.w4) {
    // one workgroup per CU (a multiple of 8 of them, so that a workgroup's tiles stay on one XCD's share of the tile
    // order) walks the tiles of all batches; never split along K
    const uint64_t all = (uint64_t)tp * tq * g.batch;
    const uint32_t slots = cus >= 8 ? cus / 8 * 8 : cus;
    plan->grid_x = (uint32_t)std::min<uint64_t>(all, slots);
    plan->grid_y = 1;
    plan->waves = (float)all / (float)cus;
    plan->workspace = 0;
    return;
  }
  if (variant == 3 && mfma_short_k(l, cus)) {
    plan->waves = (float)((double)plan->grid_x * plan->grid_y / (2.0 * cus));
    plan->grid_x = short_k_groups(cus);
    plan->grid_y = 1;
    plan->workspace = 0;
    return;
  }
  const bool eight = variant == 2 && mfma_eight_waves(l, (uint64_t)tp * tq * g.batch, cus);
  if (eight) plan->block = kMfmaEightWaves.wp * kMfmaEightWaves.wq * 64;
  const uint32_t per_cu = mfma_per_cu(l, eight ? kMfmaEightWaves : v);
  plan->waves = (float)plan->grid_x * plan->grid_y / (float)(cus * per_cu);
  plan->workspace = 0;
  const uint64_t tiles = (uint64_t)plan->grid_x * plan->grid_y;
  const uint32_t s = mfma_splits(l, v, tiles, cus, workspace_size);
  if (s > 1) {
    plan->grid_z = s;
    plan->workspace = s * tiles * v.bp * v.bq * 4;
    plan->waves = (float)tiles * s / (float)(cus * per_cu);
  }
}

// What a problem takes on a variant, in the time of one stage (128 bytes of K) of a 256 x 256 tile.  A CU holds one or a few workgroups of a
// variant at a time (mfma_per_cu()); for each such set it takes `set`, and for each workgroup the tile's area times its stages and what it
// costs around them that the others of its set do not hide (`around`, in stages) over the relative throughput of one CU inside the K
// loop (`efficiency`).  With K shared out there is a second kernel, and the partial tiles go through memory.
// Fitted to the times on every variant, weights from memory and from the caches, of 1900 int8, fp8 and bf16, 620 MXFP4 and 330 f32 problems
// (MI355X; 64 .. 32768 rows, 17 .. 12000 tokens, K = 32 .. 24000, a quarter of them in batches, workspaces of 0, 4 and 32 MiB).  What they
// pick takes 0.5 % (MXFP4 0.1 %, f32 0.2 %) more time than the best variant of each problem on average (fitted to one half 0.6, 0.3 and
// 0.5 % on the other), more than 10 % in 1.5 % of them.  With whole rounds of one workgroup per CU, fractions of a stage, shares not
// counted and one table for f32 too it was 1.5, 0.6 and 2.4 %, and short or shared K and f32 came out behind by a fifth and more: fp8
// 6608 x 2544 x 64 20.4 us on 64 x 64 tiles, 15.5 on 192 x 256; MXFP4 3980 x 3 x 8448, 4 batches 25.1 on 128 x 64 in two shares, 16.9 on
// 64 x 64; f32 17280 x 1289 x 112 80 on 256 x 256, 68 on 256 x 128.
// The variants on the 16x16 MFMA shapes (8, 9) need less energy per multiply-add, which is what bounds a GEMM that keeps the
// whole chip busy (the board sits at its power cap); on a chip that is partly idle the clock is the bound instead, so they are
// only chosen for grids that fill the chip; the same tiles at 256x128 and 128x128 measured no better than the 32x32 ones
// anywhere and are not instantiated.
struct MfmaTileCost { float efficiency, around, set; };
struct MfmaCost {
  MfmaTileCost tile[kNumMfmaVariants];
  // workgroups on a part x of the CUs take partial + (1 - partial) * x of the time of one on each: the clock is higher and memory less busy then
  float partial;
  float second_kernel;
};
static const MfmaCost kMfmaCost = {{{1.00f, 5.7f}, {0.95f, 8.5f}, {0.84f, 7.0f}, {0.64f, 1.1f, 1.87f}, {0.79f, 8.7f}, {0.46f, 0.8f, 1.44f},
                                    {0.35f, 0.5f, 1.18f}, {0.88f, 5.4f}, {1.05f, 6.1f}, {0.95f, 6.0f}, {0.37f, 2.9f}, {1.08f, 5.2f}}, 0.84f, 0.38f};
static const MfmaCost kF32Cost = {{{1.00f, 20.3f}, {0.93f, 10.2f}, {0.81f, 6.7f}, {0.62f, 0.8f, 0.36f}, {0.76f, 10.7f}, {0.64f, 1.1f, 0.90f},
                                   {0.54f, 0.5f, 0.20f}, {0.85f, 7.4f}}, 0.98f, 0.27f};  // (the others do not exist for f32)
static const MfmaCost kMxCost = {{{1.00f, 3.3f}, {0.94f, 3.2f}, {0.50f, 8.5f}, {0.61f, 0.5f, 1.26f}, {0.62f, 3.7f}, {0.44f, 1.0f, 1.05f},
                                  {0.34f, 0.4f, 1.13f}, {0.92f, 4.1f}, {}, {}, {}, {1.24f, 4.9f}}, 0.93f, 0.41f};
constexpr double kPartialTilesPerMB = 0.2;

// Skinny problems that end up with at most one 64 x 64 workgroup per CU and are not split along K are bound
// by what a CU keeps in flight: the 6-stage ring of variant 10 (80 KiB instead of 32) takes 8-17 % less time
// (bf16 14336x64x4096 29.2 us against 32.0, 4096x64x14336 71 against 87; int8 8192x64x8192 24.4 against 29.0).
static bool mfma_deep_ring(const Lowered &l, uint64_t tiles, uint32_t splits, uint32_t cus) {
  const uint32_t t = l.g.a_type;
  return t != CUDA_R_4F_E2M1 && t != CUDA_R_32F && splits == 1 && tiles <= cus && (int64_t)l.g.K * type_bits(t) / 8 >= 1536;
}

static int pick_mfma_variant(const Lowered &l, uint32_t cus, uint64_t workspace_size) {
  const GemmArgs &g = l.g;
  if (mfma_short_k(l, cus)) return 3;
  const bool swapped = g.d_si != 1;
  const uint32_t np = swapped ? g.N : g.M, nq = swapped ? g.M : g.N;
  // the tile shapes trade efficiency per CU against how evenly the problem fills the chip and what a tile costs around its K loop
  int best = 0;
  double best_cost = 0;
  for (int v = 0; v < kNumMfmaVariants; v++) {
    const MfmaVariant &t = kMfmaVariants[v];
    const uint64_t tiles = (uint64_t)ceil_div(np, t.bp) * ceil_div(nq, t.bq) * g.batch;
    if (t.stages > 4) continue;  // the deep ring: see below
    if (t.w4) {
      // The four-wave kernel, for the problems its epilogues serve, but not on a short K, where the per-tile work around the loop
      // shows: fp8 and int32 outputs from K = 2048 on (16384 x 8192 x 1024 fp8: 167 us against 153 for variant 0), int8 with
      // float outputs, f16 and bf16 from 1024 on (int8 7904 x 6288 x 1792 131 -> 99 us, bf16 5200 x 5712 x 1024 70 -> 62)
      const int epi = w4_epilogue_class(l, true);
      const bool f8 = is_f8(g.a_type);
      if (epi == W4_CLASS_NONE || g.K < (f8 || epi == W4_CLASS_I32 ? 2048 : 1024)) continue;
      if (tiles < (g.a_type == CUDA_R_8I ? ((uint64_t)cus * 3 + 3) / 4 : (uint64_t)cus)) continue;
    } else if (t.m16) {
      const bool h16 = g.a_type == CUDA_R_16F || g.a_type == CUDA_R_16BF;
      if (type_bits(g.a_type) != 8 && !h16) continue;  // the 16x16 shapes serve int8, fp8, f16 and bf16
      // power bound or not: int8 gains from three quarters of the CUs busy on.  fp8 gains little and only on
      // long runs: the 192x256 tile from two full rounds on (6144^3: 190 us against 198), the 256x256 tile
      // from four (8192^3: 405 against 408; at two rounds, 8192x4096x4096, it loses 3 %)
      // (f16 / bf16 as int8: bf16 8192^3 776 us against 840, 4096^3 102 against 108, 6144^3 336 against 360)
      const uint64_t need = (g.a_type == CUDA_R_8I || h16) ? ((uint64_t)cus * 3 + 3) / 4 : (uint64_t)cus * (t.bp == 256 ? 4 : 2);
      if (tiles < need) continue;
    }
    const bool mx = g.a_type == CUDA_R_4F_E2M1, f32 = g.a_type == CUDA_R_32F;
    const MfmaCost &c = f32 ? kF32Cost : mx ? kMxCost : kMfmaCost;
    const uint32_t s = t.w4 ? 1 : mfma_splits(l, t, tiles, cus, workspace_size);
    const int as = v == 6 && mfma_deep_ring(l, tiles, s, cus) ? 10 : v;
    const uint64_t groups = tiles * s, per_cu = mfma_per_cu(l, kMfmaVariants[as]), sets = (groups + per_cu * cus - 1) / (per_cu * cus);
    const uint64_t each = groups / cus, rem = groups % cus;
    uint32_t stages = ceil_div(ceil_div((uint32_t)((int64_t)g.K * type_bits(g.a_type) / 8), 128), s);
    if (mx && s > 1) stages = (stages + 3) / 4 * 4;  // (whole scale chunks)
    const MfmaTileCost &tc = c.tile[as];
    const double loops = (double)each + (rem ? c.partial + (1.0 - c.partial) * (double)rem / cus : 0.0);
    double cost = tc.set * (double)sets + loops * t.bp * t.bq / 65536 / tc.efficiency * (stages + tc.around);
    if (s > 1) cost += c.second_kernel + kPartialTilesPerMB * 1e-6 * (double)(s * tiles * t.bp * t.bq * 4);
    if (v == 0 || cost < best_cost) { best = v; best_cost = cost; }
  }
  return best;
}

// The 128 x 128 tile exists in both forms for 16-bit operands.  us of `groups` workgroups, n = groups / CUs of them side by
// side or in turn, u = bytes of K in a share / 4096 (bf16, MI355X, 128 to 768 tiles, K = 256 .. 1280; the choice is within 3 %
// of the better one there):
//   transposed in registers  4.6 + 1.2 n + (7.5 + 15.3 n) u
//   by the LDS reads         6.2 + 1.45 n + 2.4 per round behind the first + 27.8 u per round of two on a CU, 17.4 u for one
// -- level at K = 700 for n = 1, 430 for two, 1200 for three.  (Two stages each; the deeper ring that n = 1 has takes less: level at
// K = 704 from the caches, 10 % ahead there from memory.)  (2048 x 2048 x 128: 7.5 us in registers, 9.7 by the LDS reads;
// 3072 x 2048 x 1024: 24.3 and 20.9.)  The 256 x 256 tile is faster by the LDS reads at every K, the 64 x 64 tile beyond one stage in registers
// (K = 16 and 32: 3 to 9 % slower by the LDS reads, from the caches and from memory; 64 with one operand K-contiguous 4 and 0 %, with none 2 and 5 % faster;
// 72 to 96 with one 2 to 3 % slower from the caches and 2 to 5 % faster from memory: 2048 x 1024 x 96 A:N B:N 5.20 and 5.34, 6.28 and 5.98).
// (bf16, us from memory: 512 x 512 x 128 5.6 and 5.2, 512^3 7.9 and 6.8, 1024^3 A:N B:T 11.3 and 9.2, 2104 x 704 x 1000 16.9 and 13.8, 64 x 64 x 16384
// 70 and 48; from the caches 5.0 and 5.1, 6.7 and 6.4, 9.2 and 7.5, 11.9 and 10.7, 61 and 48.)  Another exception is
// a long operand along its row index beside up to 16 K-contiguous tokens on four to six workgroups per CU: memory bound, and the two-stage ring
// has less on its way than the registers (us from memory, in registers and by the LDS reads: 65536 x 16 x 512 17.2 and 18.7, x 2048 57 and 61, 14336 x 1 x
// 4096 in four shares 32.2 and 33.8, x 16 level; x 33 39.3 and 37.5; level at K = 64 and on eight workgroups per CU; up to three of them run
// on deeper rings: 3584 x 4 x 18944 in eight shares 38.4 and 35.3).
bool tr_lds_reads(const Lowered &l, int variant, uint64_t groups, uint32_t splits, uint32_t cus) {
  if (variant == 0 || !lds_transposable(l)) return false;
  if (variant == 2) {
    if ((uint64_t)l.g.K <= (l.a_kcontig || l.b_kcontig ? 64 : 32) * (uint64_t)std::max(splits, 1u)) return false;
    const bool a_long = l.g.M >= l.g.N, one_long = (a_long ? l.b_kcontig : l.a_kcontig) && std::min(l.g.M, l.g.N) <= 16;
    return !(one_long && groups > 3 * (uint64_t)cus && groups <= 6 * (uint64_t)cus && (uint64_t)l.g.K >= 128 * (uint64_t)std::max(splits, 1u));
  }
  if (variant == 3) return true;
  const uint64_t n = (groups + cus - 1) / std::max(cus, 1u), rounds = (n + 1) / 2;
  const double u = (double)l.g.K * 2 / 4096 / std::max(splits, 1u);
  const double regs = 4.6 + 1.2 * (double)n + (7.5 + 15.3 * (double)n) * u;
  const double lds = 6.2 + 1.45 * (double)n + 2.4 * (double)(rounds - 1) + (27.8 * (double)(n / 2) + 17.4 * (double)(n % 2)) * u;
  return lds < regs;
}

// Whether two groups of four waves of a 128 x 128 or 64 x 64 tile share a workgroup's K: at most one workgroup per CU, and enough
// stages for the gaps to matter (bf16, us: 80 x 351 x 2459, 21 batches 23.5 -> 19.1; 960 x 124 x 31971 45.6 -> 36.5; 1024 x 512 x
// 32003 76.8 -> 69; 300 x 300 x 1000 11.0 -> 9.7; level at 16 stages).  16-bit operands: f32 gains nothing, its MFMAs alone fill the time,
// and int8 0.5 us of 7.
static bool tr_two_k_groups(const Lowered &l, int variant, uint64_t groups, uint32_t splits, uint32_t cus) {
  const uint32_t t = l.g.a_type;
  if ((t != CUDA_R_16F && t != CUDA_R_16BF) || (variant != 1 && variant != 2) || groups > cus) return false;
  return (uint64_t)l.g.K * 2 / std::max(splits, 1u) >= 24 * 64;
}

static void fill_tr_plan(const Lowered &l, int variant, uint32_t cus, uint64_t workspace_size, zluda_gemm_plan *plan) {
  const GemmArgs &g = l.g;
  const TrVariant &v = kTrVariants[variant];
  const bool swapped = g.d_si != 1;
  const uint32_t np = swapped ? g.N : g.M, nq = swapped ? g.M : g.N;
  plan->variant = variant;
  plan->swapped = swapped;
  plan->grid_x = ceil_div(np, v.bp) * ceil_div(nq, v.bq); plan->grid_y = g.batch; plan->grid_z = 1;
  plan->block = v.wp * v.wq * 64;
  // workgroups that share a CU: stages of 80-byte rows, or of 128 K bytes at a pitch of 1056 bytes per KiB
  auto per_cu_of = [&](bool by_lds, uint64_t stages) { return (uint32_t)std::min<uint64_t>(160u * 1024u / (stages * (v.bp + v.bq) * (by_lds ? 132u : 80u)), 4u); };
  // (two stages each: what the rule below was measured with, and the least that any form has)
  const uint32_t per_cu = per_cu_of(tr_lds_reads(l, variant, (uint64_t)plan->grid_x * plan->grid_y, 1, cus), 2);
  plan->workspace = 0;
  // Split-K as for the K-contiguous kernels: grid_z workgroups share a tile's K range through the
  // caller's workspace when K is long enough (`least`) and the tiles leave half of the chip idle --
  // half of the CUs, or, for skinny problems (<= 64 rows or columns: memory bound, a workgroup keeps
  // only ~16 KiB in flight), half of the workgroup slots.  N-contiguous weights, 16 tokens, us:
  // 4096x14336 89 -> 25, 4096x4096 31 -> 14, 14336x4096 31 -> 24; 14336x128x4096 would lose (37 -> 42).
  const uint64_t tiles = (uint64_t)plan->grid_x * plan->grid_y;
  const uint64_t slots = (uint64_t)cus * per_cu;
  const bool skinny = std::min(g.M, g.N) <= 64;
  const uint64_t kbytes = (uint64_t)g.K * type_bits(g.a_type) / 8;
  // Where the loop that gets shorter outweighs the second kernel and the partial tiles' way through memory depends on both, us whole and in
  // as many shares as there can be: f32 256 x 256 x 384 9.3 and 8.2, 512 x 512 x 384 9.4 and 10.1, x 1024 19.0 and 14.3; bf16 256 x 256 x 1024
  // 8.7 and 8.5, 512 x 512 x 1024 8.9 and 10.0, x 2048 12.9 and 12.8; int8 300 x 300 x 1088 8.3 and 9.3, x 1536 10.2 and 9.0, 512 x 512 x 1088
  // 7.2 and 10.1, x 2048 10.7 and 10.5.  The lines lie at the least K that gains on few tiles; 8-bit operands gain from 1300 to 2500 bytes
  // on, and are split from 17 stages on as they have been.  (Choosing the number of shares by such a cost gained 2 % over 392 problems whose operands
  // were in the caches and none where they were not, and lost up to 20 % on some.)
  const uint64_t least = skinny ? 1024 : g.a_type == CUDA_R_32F ? 1536 : type_bits(g.a_type) == 16 ? 2048 : 1088;
  if (tiles * 2 <= (skinny ? slots : (uint64_t)cus) && kbytes >= least && (uint64_t)ceil_div(np, v.bp) * v.bp <= (1u << 20)) {
    uint32_t s = (uint32_t)std::min<uint64_t>({8, slots / tiles, kbytes / 512});
    const uint64_t per_split = (uint64_t)g.batch * ceil_div(np, v.bp) * v.bp * ceil_div(nq, v.bq) * v.bq * 4;
    while (s > 1 && s * per_split > workspace_size) s--;
    if (s > 1) {
      plan->grid_z = s;
      plan->workspace = s * per_split;
    }
  }
  const uint64_t groups = tiles * plan->grid_z;
  const bool lds_reads = tr_lds_reads(l, variant, groups, plan->grid_z, cus);
  if (!lds_reads && tr_two_k_groups(l, variant, groups, plan->grid_z, cus)) plan->block = 512;
  plan->waves = (float)groups / (float)(cus * per_cu_of(lds_reads, lds_reads ? tr_ring_stages(variant, groups, cus) : 2));
}

// Tile choice of the transposing kernel.  A CU runs up to `per_cu` workgroups of a variant side by
// side; the time it needs for n of them (same K) was measured on MI355X (int8, K = 4096, us):
// 256x256: 71;  128x128: 37 alone, 48 for two;  64x64: 22 alone, 40 for four  ->  base + slope * n.
// Cost of a variant = full rounds x time(per_cu) + time(what is left per CU).
struct TrCost { uint32_t per_cu; float base, slope; };
static const TrCost kTrCost[kNumTrVariants] = {{1, 0.0f, 71.0f}, {2, 26.0f, 11.0f}, {4, 16.0f, 6.0f}, {1, 0.0f, 67.0f}};

// f16 and bf16: the split along K that the variant would get counts as well, and where the LDS reads transpose
// (tr_lds_reads()) the variants 1 and 3 have times of their own (kTrCostLds).  us for 4096 bytes of K:
// 128x128 25 + 3.3 n, 256x256 53 on a full chip (8192 x 4096 x 2048 121 us against 174 on 128x128; 2048 x 4096 x 8192, 128
// tiles, 164 against 130); the others as above.  Around the loop 4 us, and for a split the second kernel and the partial
// tiles' way through memory at 3 TB/s.  (The variants 1 and 2 by the LDS reads take less than that by now, both alike, and variant 2 is left
// with its time in registers: over 300 problems of 128 to 4096 rows and columns and K = 128 to 8192 what these pick takes 0.3 % more time than the best
// variant on average with operands from memory, 1.3 % from the caches; more than 10 % in 2 and 11 of them: 1376 x 448 x 3000 A:N B:T from the caches 22.5 us
// on 128 x 128 tiles, 13.7 on 64 x 64.)
// (1024 x 512 x 1024 on 128x128 would take 20 us split, 64x64 take 10).
static const TrCost kTrCostLds[kNumTrVariants] = {{1, 0.0f, 71.0f}, {2, 25.0f, 3.3f}, {4, 16.0f, 6.0f}, {1, 0.0f, 53.0f}};

static int pick_tr_variant_h16(const Lowered &l, uint32_t cus, uint64_t workspace_size) {
  const double units = (double)l.g.K * 2 / 4096;
  int best = 0;
  double best_cost = 0;
  for (int v = 0; v < kNumTrVariants; v++) {
    zluda_gemm_plan p;
    memset(&p, 0, sizeof(p));
    fill_tr_plan(l, v, cus, workspace_size, &p);
    const uint64_t groups = (uint64_t)p.grid_x * p.grid_y * p.grid_z;
    const bool lds = tr_lds_reads(l, v, groups, p.grid_z, cus);
    const TrCost &c = (lds ? kTrCostLds : kTrCost)[v];
    const uint64_t slots = (uint64_t)cus * c.per_cu;
    if (kTrVariants[v].m16 && !lds && groups * 4 < (uint64_t)cus * 3) continue;
    const uint64_t full = groups / slots, rem = groups % slots;
    double cost = (double)full * (c.base + c.slope * c.per_cu);
    if (rem) cost += c.base + c.slope * (double)((rem + cus - 1) / cus);
    cost = 4.0 + cost * units / p.grid_z;
    if (p.grid_z > 1) cost += 4.0 + (double)p.workspace * 2 / 3e6;
    if (v == 0 || cost < best_cost) { best = v; best_cost = cost; }
  }
  return best;
}

static int pick_tr_variant(const Lowered &l, uint32_t cus, uint64_t workspace_size) {
  const GemmArgs &g = l.g;
  if (g.a_type == CUDA_R_16F || g.a_type == CUDA_R_16BF) return pick_tr_variant_h16(l, cus, workspace_size);
  const bool swapped = g.d_si != 1;
  const uint32_t np = swapped ? g.N : g.M, nq = swapped ? g.M : g.N;
  int best = 0;
  double best_cost = 0;
  for (int v = 0; v < kNumTrVariants; v++) {
    const TrVariant &t = kTrVariants[v];
    const TrCost &c = kTrCost[v];
    const uint64_t tiles = (uint64_t)ceil_div(np, t.bp) * ceil_div(nq, t.bq) * g.batch;
    // the 16x16 shape: int8, f16 and bf16, and only where the chip is full enough to sit at its power cap
    const bool m16_type = g.a_type == CUDA_R_8I || g.a_type == CUDA_R_16F || g.a_type == CUDA_R_16BF;
    if (t.m16 && (!m16_type || tiles * 4 < (uint64_t)cus * 3)) continue;
    const uint64_t slots = (uint64_t)cus * c.per_cu;
    const uint64_t full = tiles / slots, rem = tiles % slots;
    double cost = (double)full * (c.base + c.slope * c.per_cu);
    if (rem) cost += c.base + c.slope * (double)((rem + cus - 1) / cus);
    if (v == 0 || cost < best_cost) { best = v; best_cost = cost; }
  }
  return best;
}

// Enough shares for about four workgroups per CU at 64 rows a workgroup, 64 terms at the least in each: 2048 sums of 4096 terms
// take 1024 workgroups in 32 shares on 256 CUs.  (A workgroup takes 16 bytes' worth of rows per lane: with K shared out 32 to 128
// of an operand, 128 or 256 of a GELU gradient; unshared half of the former and 16 or 32.)
uint32_t row_sum_shares(int64_t rows, int64_t len, int64_t batch, uint64_t workspace_size, uint32_t cus) {
  const int64_t groups = (rows + 63) / 64 * batch;
  int64_t s = std::min<int64_t>({(4 * (int64_t)cus + groups - 1) / groups, len / 64, 65535});
  const uint64_t per_share = (uint64_t)rows * batch * 4;
  if (s > 1 && (uint64_t)s * per_share > workspace_size) s = (int64_t)(workspace_size / per_share);
  return s > 1 ? (uint32_t)s : 1u;
}

// scratch the bias-gradient sums of the problem would use, within `workspace_size`
static uint64_t row_sum_workspace(const GemmArgs &g, uint64_t workspace_size, uint32_t cus) {
  int64_t rows = 0, len = 0;
  if (g.bgrad_src == 1 && g.a_sk > g.a_si) { rows = g.M; len = g.K; }
  else if (g.bgrad_src == 2 && g.b_sk > g.b_sj) { rows = g.N; len = g.K; }
  else if (g.aux_bgrad && g.d_si == 1) { rows = g.M; len = g.N; }
  if (rows == 0) return 0;
  const uint32_t s = row_sum_shares(rows, len, g.batch, workspace_size, cus);
  return s > 1 ? (uint64_t)s * rows * g.batch * 4 : 0;
}

// The forms the epilogues with an aux matrix are instantiated for: 16-bit operands on the tile kernels up to a size of the wave tile, unsplit,
// 16-bit D and aux that the 16-byte stores of eight rows fit.  us with a pass behind the matmul and without (bf16, operands in the caches):
// 8192 x 4096 x 2048 GELU_AUX_BIAS 122 -> 110, A:N B:N DGELU_BGRAD 152 -> 138; 2048 x 1000 x 1024 13.2 -> 10.1 and 21.1 -> 13.4; 1000 x 700 x 496
// 9.0 -> 7.1 and 16.5 -> 12.2.
bool aux_in_epilogue(const Lowered &l, const zluda_gemm_plan &plan, bool dry) {
  const GemmArgs &g = l.g;
  if (!g.aux_mode || (plan.kernel != ZLUDA_KERNEL_MFMA_H16 && plan.kernel != ZLUDA_KERNEL_MFMA_TR16)) return false;
  if (g.d_type != CUDA_R_16F && g.d_type != CUDA_R_16BF) return false;
  if (plan.grid_z > 1 || plan.swapped || g.d_si != 1 || g.aux_si != 1) return false;
  if (g.beta_mode != SCALAR_VALUE || (!dry && g.beta_val.f != 0.0f)) return false;
  if (g.alpha_mode == VECTOR_DEV || g.a_scale_mode == SCALE_OUTER_VEC || g.b_scale_mode == SCALE_OUTER_VEC) return false;
  if (g.M & 7) return false;
  const int64_t pitches = g.d_sj | g.aux_sj | (g.batch > 1 ? g.d_sb | g.aux_sb : 0);
  if ((pitches & 7) || g.d_sj >= kNarrowPitch || g.aux_sj >= kNarrowPitch) return false;
  if (!dry && (((uintptr_t)g.D | (uintptr_t)g.aux) & 15)) return false;
  if (plan.kernel == ZLUDA_KERNEL_MFMA_H16) {
    if (plan.variant >= (uint32_t)kNumMfmaVariants) return false;
    const MfmaVariant &v = kMfmaVariants[plan.variant];
    // (the gradient: of operands that are not K-contiguous; D's scale is folded into GELU's reciprocal there, which makes NaN of large inputs
    // where the scale is zero)
    if (v.w4) return g.aux_mode == 1 && !g.d_scale && w4_epilogue_class(l, dry) == W4_CLASS_BF16;
    const MfmaVariant &w = plan.variant == 2 && plan.block == 512 ? kMfmaEightWaves : v;
    // (not the short-K form, whose workgroups walk the tiles of all batches: as many of them as one batch has tiles, with 512 of those)
    return plan.grid_x == ceil_div(g.M, v.bp) * ceil_div(g.N, v.bq) && plan.grid_y == (uint32_t)g.batch &&
           (v.m16 || aux_on_wave_tile32(w.bp / w.wp, w.bq / w.wq));
  }
  if (plan.variant >= (uint32_t)kNumTrVariants) return false;
  const TrVariant &t = kTrVariants[plan.variant];
  return t.m16 || aux_on_wave_tile32(t.bp / t.wp, t.bq / t.wq);
}

uint32_t aux_sum_shares(const Lowered &l, const zluda_gemm_plan &plan) {
  if (plan.kernel == ZLUDA_KERNEL_MFMA_H16) return ceil_div(l.g.N, kMfmaVariants[plan.variant].bq) * kMfmaVariants[plan.variant].wq;
  return ceil_div(l.g.N, kTrVariants[plan.variant].bq) * kTrVariants[plan.variant].wq;
}

uint32_t transposing_under_generic(const Lowered &l) {
  const uint32_t family = transposing_family(l, true);
  if (!family || transposing_family(l, false)) return 0;
  for (uint32_t k : {ZLUDA_KERNEL_MFMA_I8, ZLUDA_KERNEL_MFMA_F8, ZLUDA_KERNEL_MFMA_H16, ZLUDA_KERNEL_MFMA_F32})
    if (family_supports(k, l)) return 0;
  return family;
}

// Workgroups of the slab kernel per batch: at most one per CU (its LDS ring fills the CU), more only when the rows would not fit
// into 4 blocks per workgroup otherwise.
// (a short block costs its workgroup as many DMA instructions as a full one: the fewest rounds of blocks that
// fit the CUs, shared out evenly -- 896 blocks on 256 CUs: 224 workgroups x 4)
static uint32_t slab_groups(uint32_t rows, uint32_t cus) {
  const uint32_t nrb = ceil_div(rows, 16);
  return std::max(ceil_div(nrb, ceil_div(nrb, cus)), ceil_div(rows, 64));
}

static void fill_decode_plan(const Lowered &l, int variant, uint32_t cus, zluda_gemm_plan *plan) {
  const GemmArgs &g = l.g;
  const DecodeVariant &v = kDecodeVariants[variant];
  const bool swapped = g.M < g.N;  // weights are the long operand
  const uint32_t rows = swapped ? g.N : g.M;
  const uint32_t nrb = ceil_div(rows, 16);
  // Stream kernel: 8 waves x 2 slots x 4 KiB = 64 KiB in flight per CU is the measured optimum on
  // MI355X (14.8 us for 58.7 MB; 128 KiB in flight: 15.8-16.8 us, 32 KiB: 15.9 us), so one 8-wave
  // workgroup per CU, two 4-wave ones.
  const uint32_t resident = v.stream == 2 ? cus : v.stream ? cus * (v.nw == 8 ? 1 : 2) : cus * (v.nw == 8 ? 2 : 4);
  uint32_t grid;
  if (v.stream == 2) grid = slab_groups(rows, cus);
  else if (v.stream) grid = std::min(nrb, resident);  // contiguous, balanced row ranges
  else grid = nrb <= resident ? nrb : ceil_div(nrb, ceil_div(nrb, resident));
  plan->variant = variant;
  plan->swapped = swapped;
  plan->grid_x = grid; plan->grid_y = g.batch; plan->grid_z = 1;
  plan->block = v.nw * 64;
  plan->waves = (float)grid * g.batch / (float)resident;
  plan->workspace = 0;
}

static int pick_decode_variant(const Lowered &l, uint32_t cus) {
  const int K = l.g.K;
  // the slab form where it applies and one workgroup per CU holds the rows (14336 x 16 x 4096 int8: 12.4 us
  // against 14.8 for the stream kernel proper)
  // (two token blocks on one unit per slab, variant 20, only up to two blocks of rows per CU: 4096 x 32 x 4096
  // 8.9 us against 10.0, but 14336 x 32 x 4096 18.1 against 16.7; with two units, variant 17, it wins
  // throughout: 8192 x 32 x 8192 15.4 against 22.0)
  const uint32_t rows = (uint32_t)std::max(l.g.M, l.g.N);
  const bool h16 = l.g.a_type == CUDA_R_16F || l.g.a_type == CUDA_R_16BF;
  const bool mx = l.g.a_type == CUDA_R_4F_E2M1;
  // Beyond 64 rows per CU the workgroups take more than one round, each of which costs what a shape's whole cover of K does, however
  // little of it the problem has.  (us on slabs and on the best MFMA tiles, weights from memory.  A loop over one matrix of less than
  // 200 MB finds it in the memory-side cache, which the tiles gain more from: 20480 x 4 x 4096 33 and 26, 32768 x 4 x 3072 33 and 30.)
  //   16-bit weights: with K beyond 4096 always (bf16 28672 x 16 x 8192 80 and 99).  Up to 8 tokens, K that fills the cover (18000 x 4 x 2048
  //   18.6 and 21.3, 20480 x 4 x 4096 33.7 and 40.2), or five eighths of the 8-wave one (26000 x 4 x 2560 26.2 and 28.4, 18000 x
  //   4 x 3584 29.9 and 32.5, 37888 x 4 x 3584 48.3 and 59.4; but 18000 x 4 x 2304 23.4 and 21.5, 50000 x 4 x 1408 33.9 and 29.3).
  //   MXFP4: rounds that are 70 % full (57344 x 4 x 8192 in 3.5 42.7 and 56.5, but 20480 x 8 x 5120 in 1.25 17.6 and 17.3) and K that fills three
  //   quarters of the cover (28672 x 4 x 6144 19.0 and 21.2, 43000 x 4 x 12288 48.8 and 67.6; but 28672 x 4 x 4352 17.1 and 15.3), all of it with two
  //   token blocks (43000 x 24 x 8192 40.7 and 54.2; but 28672 x 24 x 5120 19.9 and 18.6).
  const uint64_t round = 64 * (uint64_t)cus;
  auto rounds_ok = [&](int v) {
    const int cover = kDecodeVariants[v].nw * kDecodeVariants[v].steps * 64, tokens = std::min(l.g.M, l.g.N);
    const int64_t kb = (int64_t)K * type_bits(l.g.a_type) / 8;
    if (rows <= round) return true;
    if (mx) return (uint64_t)rows * 10 >= (rows + round - 1) / round * round * 7 && (tokens > 16 ? kb == cover : kb * 4 >= cover * 3);
    return h16 && (kb > 8192 || (tokens <= 8 && (kb == cover || kb * 8 >= 8192 * 5)));
  };
  // (MXFP4 in batches: a workgroup fetches the activations for as few as 16 rows, and with more than two of them per CU the MFMA tiles
  // are ahead unless K is long: us on slabs and on tiles, weights from memory, 428 x 25 x 4608, 64 batches, 1728 workgroups 40.4 and 17.0,
  // 4012 x 16 x 9216, 8, 2008 48 and 30, 9000 x 15 x 8704, 3, 564 31.5 and 26.3; 252 x 2 x 10496, 32, 512 13.1 and 15.7, 828 x 8 x 12288, 8,
  // 416 13.5 and 17.2, 192 x 5 x 7936, 16, 192 7.4 and 16.2; 15804 x 10 x 11520, 3, 741 51 and 66, 552 x 16 x 23296, 32, 1120 51 and 58)
  const bool few_groups = !mx || l.g.batch == 1 || K >= 11264 || (uint64_t)slab_groups(rows, cus) * l.g.batch <= 2 * (uint64_t)cus;
  for (int v = 0; v < kNumDecodeVariants; v++)
    if (kDecodeVariants[v].stream == 2 && decode_variant_ok(l, v) && rounds_ok(v) && few_groups &&
        !(kDecodeVariants[v].steps == 8 && rows > 32 * cus && !mx))
      return v;
  // the stream instantiation with the least cover that takes K
  int best = -1;
  for (int v = 0; v < kNumDecodeVariants; v++)
    if (kDecodeVariants[v].stream == 1 && decode_variant_ok(l, v) &&
        (best < 0 || kDecodeVariants[v].nw * kDecodeVariants[v].steps < kDecodeVariants[best].nw * kDecodeVariants[best].steps))
      best = v;
  if (best >= 0) return best;
  for (int v = 0; v < kNumDecodeVariants; v++)
    if (!kDecodeVariants[v].stream && K == kDecodeVariants[v].nw * kDecodeVariants[v].steps * 64 && decode_variant_ok(l, v))
      return v;
  return 0;
}

} // namespace zluda_amd

using namespace zluda_amd;

extern "C" uint32_t zluda_gemm_variant_count(uint32_t kernel) {
  switch (kernel) {
  case ZLUDA_KERNEL_GENERIC: return 1;
  case ZLUDA_KERNEL_MFMA_I8: case ZLUDA_KERNEL_MFMA_F8: return kNumMfmaVariants;
  case ZLUDA_KERNEL_MFMA_H16: return kNumMfmaVariantsH16;
  case ZLUDA_KERNEL_MFMA_F32: return kNumMfmaVariants32;  // the 16x16-shape ones serve int8, fp8, f16 and bf16
  case ZLUDA_KERNEL_MFMA_MXF4: return kNumMfmaVariants;   // (the eight 32x32-shape ones and the four-wave kernel; those between are refused)
  case ZLUDA_KERNEL_DECODE_W8A8: return kNumDecodeVariants;
  case ZLUDA_KERNEL_MFMA_TR8: case ZLUDA_KERNEL_MFMA_TR16: return kNumTrVariants;
  case ZLUDA_KERNEL_MFMA_TR32: return kNumTrVariants - 1;  // the 16x16-shape one is not instantiated for f32
  default: return 0;
  }
}

extern "C" uint32_t zluda_gemm_plan_problem(const zluda_gemm_problem *p, uint32_t forced_kernel,
                                            int32_t forced_variant, uint32_t cu_count,
                                            zluda_gemm_plan *plan) {
  if (!plan) return CUBLAS_STATUS_INVALID_VALUE;
  Lowered l;
  // planning never dereferences data: NULL pointers mean "aligned as the preferences promise"
  uint32_t st = lower_problem(p, true, &l);
  if (st) return st;
  if (cu_count == 0) cu_count = 256;
  memset(plan, 0, sizeof(*plan));
  uint32_t kernel = forced_kernel;
  if (kernel == ZLUDA_KERNEL_AUTO) {
    static const uint32_t order[] = {ZLUDA_KERNEL_DECODE_W8A8, ZLUDA_KERNEL_MFMA_I8, ZLUDA_KERNEL_MFMA_F8,
                                     ZLUDA_KERNEL_MFMA_MXF4, ZLUDA_KERNEL_MFMA_H16, ZLUDA_KERNEL_MFMA_TR8,
                                     ZLUDA_KERNEL_MFMA_TR16, ZLUDA_KERNEL_MFMA_F32, ZLUDA_KERNEL_MFMA_TR32, ZLUDA_KERNEL_GENERIC};
    for (uint32_t k : order) {
      if (!family_supports(k, l)) continue;
      if (k == ZLUDA_KERNEL_DECODE_W8A8) {
        // (some variant takes the problem, but not necessarily the one the rules below pick for this chip: 16-bit
        // weights have the slab form only, which is given at most 64 rows per CU)
        if (!decode_variant_ok(l, pick_decode_variant(l, cu_count))) continue;
        const int tokens = std::min(l.g.M, l.g.N);
        const bool stream = kDecodeVariants[pick_decode_variant(l, cu_count)].stream;
        if (tokens > (stream ? kDecodeAutoMaxTokensStream : kDecodeAutoMaxTokens)) continue;
        // three token blocks only up to 32 rows per CU: beyond, 64-wide tiles read the weights as fast
        // (14336 x 48 x 4096 int8: 17.0 us against 20.7; 8192 x 33 x 4096: 14.0 against 13.9)
        if (tokens > 32 && (uint32_t)std::max(l.g.M, l.g.N) > 32 * cu_count) continue;
      }
      if (k == ZLUDA_KERNEL_DECODE_W8A8 && !kDecodeVariants[pick_decode_variant(l, cu_count)].stream &&
          family_supports(ZLUDA_KERNEL_MFMA_I8, l)) {  // (int8 only: fp8 has no such variant)
        // K outside the stream kernel's table: the register-streaming variant measures slower than
        // 64x64 MFMA tiles (split along K when the workspace allows) as soon as those give at
        // least half of the CUs a workgroup (5120x16x13824: 37 us against 23; 18944x32x3584: 46
        // against 25; but 2048x16x2560, 32 tiles: 8 against 12)
        zluda_gemm_plan mfma;
        memset(&mfma, 0, sizeof(mfma));
        fill_mfma_plan(l, pick_mfma_variant(l, cu_count, p->workspace_size), cu_count, p->workspace_size, &mfma);
        if ((uint64_t)mfma.grid_x * mfma.grid_y * mfma.grid_z * 2 >= cu_count) continue;
      }
      kernel = k;
      break;
    }
  } else if (!family_supports(kernel, l)) {
    return CUBLAS_STATUS_NOT_SUPPORTED;
  }
  plan->kernel = kernel;
  switch (kernel) {
  case ZLUDA_KERNEL_GENERIC:
    plan->variant = 0; plan->swapped = 0;
    plan->grid_x = ceil_div(l.g.M, 64); plan->grid_y = ceil_div(l.g.N, 64); plan->grid_z = l.g.batch;
    plan->block = 256;
    plan->waves = (float)plan->grid_x * plan->grid_y * plan->grid_z / (float)(cu_count * 8);
    if (plan->grid_y > 65535) return CUBLAS_STATUS_NOT_SUPPORTED;
    // what only alignment or a ragged K keeps from the transposing kernel runs on it all the same: variant 1 + v
    if (transposing_under_generic(l)) {
      fill_tr_plan(l, pick_tr_variant(l, cu_count, p->workspace_size), cu_count, p->workspace_size, plan);
      plan->variant++;
    }
    break;
  case ZLUDA_KERNEL_MFMA_I8: case ZLUDA_KERNEL_MFMA_F8: case ZLUDA_KERNEL_MFMA_MXF4: case ZLUDA_KERNEL_MFMA_H16:
  case ZLUDA_KERNEL_MFMA_F32: {
    int v = forced_variant >= 0 ? forced_variant : pick_mfma_variant(l, cu_count, p->workspace_size);
    const bool w4 = v < kNumMfmaVariants && kMfmaVariants[v].w4;
    if (v >= kNumMfmaVariants || (v >= kNumMfmaVariants32 && !w4 && kernel != ZLUDA_KERNEL_MFMA_I8 && kernel != ZLUDA_KERNEL_MFMA_F8 &&
                                  kernel != ZLUDA_KERNEL_MFMA_H16) || (v >= kNumMfmaVariantsH16 && kernel == ZLUDA_KERNEL_MFMA_H16) ||
        (w4 && kernel == ZLUDA_KERNEL_MFMA_F32))
      return CUBLAS_STATUS_INVALID_VALUE;
    // the four-wave kernel exists for int8, for fp8 without block scales, for MXFP4, for f16 and for bf16
    if (w4 && !(l.g.a_type == CUDA_R_8I || kernel == ZLUDA_KERNEL_MFMA_F8 ||
                (l.g.a_type == CUDA_R_4F_E2M1 && l.g.b_type == CUDA_R_4F_E2M1) ||
                ((l.g.a_type == CUDA_R_16F || l.g.a_type == CUDA_R_16BF) && l.g.b_type == l.g.a_type)))
      return CUBLAS_STATUS_NOT_SUPPORTED;
    fill_mfma_plan(l, v, cu_count, p->workspace_size, plan);
    if (forced_variant < 0 && v == 6 && mfma_deep_ring(l, (uint64_t)plan->grid_x * plan->grid_y, plan->grid_z, cu_count))
      fill_mfma_plan(l, 10, cu_count, 0, plan);
    break;
  }
  case ZLUDA_KERNEL_MFMA_TR8: case ZLUDA_KERNEL_MFMA_TR16: case ZLUDA_KERNEL_MFMA_TR32: {
    int v = forced_variant >= 0 ? forced_variant : pick_tr_variant(l, cu_count, p->workspace_size);
    if (v >= kNumTrVariants || (kTrVariants[v].m16 && l.g.a_type != CUDA_R_8I && l.g.a_type != CUDA_R_16F && l.g.a_type != CUDA_R_16BF))
      return CUBLAS_STATUS_INVALID_VALUE;
    fill_tr_plan(l, v, cu_count, p->workspace_size, plan);
    break;
  }
  case ZLUDA_KERNEL_DECODE_W8A8: {
    int v = forced_variant >= 0 ? forced_variant : pick_decode_variant(l, cu_count);
    if (v >= kNumDecodeVariants) return CUBLAS_STATUS_INVALID_VALUE;
    // (asked for by name: the variant that takes the problem, also where the rules above leave it to another family)
    for (int n = 0; forced_variant < 0 && n < kNumDecodeVariants && !decode_variant_ok(l, v); n++) v = n;
    if (!decode_variant_ok(l, v)) return CUBLAS_STATUS_NOT_SUPPORTED;
    fill_decode_plan(l, v, cu_count, plan);
    break;
  }
  default: return CUBLAS_STATUS_NOT_SUPPORTED;
  }
  // (the sums run behind the matmul and its reduction, in the same scratch)
  plan->workspace = std::max(plan->workspace, row_sum_workspace(l.g, p->workspace_size, cu_count));
  if (l.g.aux_bgrad && aux_in_epilogue(l, *plan, true)) {
    const uint64_t sums = (uint64_t)aux_sum_shares(l, *plan) * l.g.M * l.g.batch * 4;
    if (sums <= p->workspace_size) plan->workspace = std::max(plan->workspace, sums);
  }
  return CUBLAS_STATUS_SUCCESS;
}
