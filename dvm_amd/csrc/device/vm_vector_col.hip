// gfx950 vector VM, column build (VS_COLS in isa_gfx950.h): programs that load one operand, reduce it along its outer axis
// and store what follows per output: a column sum (the bias gradient of a linear layer), a column maximum, the first launch
// of a batch-norm over channels-last data.
//
// What bounds such a program is how many bytes its few workgroups have in flight. The generic kernel gives a workgroup 512
// columns, so a [489, 824] operand ran on two of 256 compute units, and where the columns do not fill its waves every load
// went element by element: 100 us, now 7. Here a workgroup owns the columns of one 128-byte line,
// its lanes stand tx along them and the rest along the rows, and every lane has 8 or 16 rows in flight at once. Lanes past
// the last column, and the lane that holds a ragged end, take the last eight columns instead and store the same values.
// Partials accumulate in fp64 per column, rows in ascending order per lane, then across the lanes and waves in a fixed order.
#include "vec_common.h"

#pragma clang fp contract(off)  // (every instruction rounds its own result, as on the other builds)

namespace {

__shared__ __align__(16) uint32_t prog_lds[DVM_PARAM_BYTES / 4];

typedef uint32_t vu4_any __attribute__((ext_vector_type(4), aligned(2)));  // 16 bytes at any address of a 16- or 32-bit element

struct ColAcc {
  double v[E];
};

template <int KIND, bool SQUARE>
__device__ __forceinline__ void col_add(ColAcc &r, const float (&x)[E]) {
  FOR_E r.v[e] = red_op<KIND>(r.v[e], static_cast<double>(SQUARE ? x[e] * x[e] : x[e]));
}
// what a reduce slot does with one row's eight values; how: its kind, and whether it sums squares
__device__ __forceinline__ void col_row(ColAcc &r, uint32_t how, const float (&x)[E]) {
  switch (how) {
    case VR_SUM: col_add<VR_SUM, false>(r, x); break;
    case VR_SUM | VRF_SQUARE: col_add<VR_SUM, true>(r, x); break;
    case VR_MAX: col_add<VR_MAX, false>(r, x); break;
    default: col_add<VR_MIN, false>(r, x); break;
  }
}

constexpr uint32_t kNoSlot = 0xffffffffu;

// NR rows, `step` bytes apart, that start at `at`; rows from row `left` on are past the end (they fetch the first row again and
// count for nothing). F32: 32-bit elements.
template <int NR, bool F32, bool GUARD>
__device__ __forceinline__ void col_rows(uint64_t at, uint64_t step, uint32_t left, uint32_t dtype, uint32_t how0, uint32_t how1, ColAcc &r0, ColAcc &r1) {
  vu4 a[NR], b[F32 ? NR : 1];
#pragma unroll
  for (int j = 0; j < NR; ++j) {
    const uint64_t p = (!GUARD || static_cast<uint32_t>(j) < left) ? at + static_cast<uint32_t>(j) * step : at;
    a[j] = *reinterpret_cast<const DVM_GLOBAL vu4_any *>(p);
    if constexpr (F32) b[j] = *reinterpret_cast<const DVM_GLOBAL vu4_any *>(p + 16);
  }
#pragma unroll
  for (int j = 0; j < NR; ++j) {
    float x[E];
    if constexpr (F32) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[i] = __uint_as_float(a[j][i]);
        x[4 + i] = __uint_as_float(b[j][i]);
      }
    } else if (dtype == VDT_BF16) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[2 * i] = __uint_as_float(a[j][i] << 16);
        x[2 * i + 1] = __uint_as_float(a[j][i] & 0xffff0000u);
      }
    } else {
      const vh8 h = __builtin_bit_cast(vh8, a[j]);
      FOR_E x[e] = static_cast<float>(h[e]);
    }
    if (!GUARD || static_cast<uint32_t>(j) < left) {
      if (how0 != kNoSlot) col_row(r0, how0, x);
      if (how1 != kNoSlot) col_row(r1, how1, x);
    }
  }
}

// Combines the partials of the lanes that stand along the rows: across the rows of a wave by shuffles, across the waves
// through local memory; the first tx lanes of the workgroup end up with the results.
__device__ __forceinline__ void col_combine(ColAcc &r, uint32_t kind, uint32_t tlog, uint32_t tid, uint32_t nthreads) {
  const uint32_t tx = 1u << tlog, lane = tid & 63u;
  for (uint32_t d = tx; d < 64u; d <<= 1) FOR_E r.v[e] = red_combine(kind, r.v[e], __shfl_xor(r.v[e], static_cast<int>(d), 64));
  if (nthreads <= 64u) return;
  if (lane < tx) FOR_E lds[((tid >> 6) * tx + lane) * E + e] = r.v[e];
  __syncthreads();
  for (uint32_t t = tid; t < tx * E; t += nthreads) {
    double s = lds[t];
    for (uint32_t w = 1; w < nthreads >> 6; ++w) s = red_combine(kind, s, lds[w * tx * E + t]);
    lds[t] = s;
  }
  __syncthreads();
  if (tid < tx) FOR_E r.v[e] = lds[tid * E + e];
  __syncthreads();
}

__device__ __forceinline__ void col_store(const VMemDesc &m, uint64_t off, const float (&v)[E]) {
  if (m.flags & VMF_GATHER) {
    const uint64_t step = m.flags >> 8;
    FOR_E {
      const uint64_t at = off + static_cast<uint64_t>(e) * step;
      if (m.dtype == VDT_F32) reinterpret_cast<DVM_GLOBAL float *>(m.addr)[at] = v[e];
      else if (m.dtype == VDT_F16) reinterpret_cast<DVM_GLOBAL _Float16 *>(m.addr)[at] = static_cast<_Float16>(v[e]);
      else reinterpret_cast<DVM_GLOBAL uint16_t *>(m.addr)[at] = static_cast<uint16_t>(f32_to_bf16_bits(v[e]));
    }
    return;
  }
  if (m.dtype == VDT_F32) {
    DVM_GLOBAL vu4_any *p = reinterpret_cast<DVM_GLOBAL vu4_any *>(m.addr + off * 4u);
    p[0] = vu4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])};
    p[1] = vu4{__float_as_uint(v[4]), __float_as_uint(v[5]), __float_as_uint(v[6]), __float_as_uint(v[7])};
  } else if (m.dtype == VDT_BF16) {
    *reinterpret_cast<DVM_GLOBAL vu4_any *>(m.addr + off * 2u) = vu4{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7])};
  } else {
    vh8 h;
    FOR_E h[e] = static_cast<_Float16>(v[e]);
    *reinterpret_cast<DVM_GLOBAL vu4_any *>(m.addr + off * 2u) = __builtin_bit_cast(vu4, h);
  }
}

}  // namespace

extern "C" __global__ void __launch_bounds__(512) dvm_vm_vec_col(const VmParam p) {
  const uint32_t tid = threadIdx.x, nthreads = blockDim.x;
  fetch_program(prog_lds, p.w, [&]() { return (prog_lds[offsetof(VVecHeader, code_off) / 4] + prog_lds[offsetof(VVecHeader, n_code) / 4]) * 2; });
#define HDR(field) uni(prog_lds[offsetof(VVecHeader, field) / 4])
  const VDim *kdims = reinterpret_cast<const VDim *>(prog_lds + offsetof(VVecHeader, kdims) / 4);
  const uint32_t n_kdim = HDR(n_kdim), n_kidx = HDR(n_kidx), n_items = HDR(n_items), mem_off = HDR(mem_off);
  const uint32_t *code = prog_lds + 2u * HDR(code_off);
  auto desc_of = [&](uint32_t a) { return load_desc(prog_lds, mem_off, a); };
  // [sweep] [load] [one or two reduces], then the arithmetic on the results
  const VMemDesc m = desc_of(uni(code[2]) >> 24);
  uint32_t how0 = kNoSlot, how1 = kNoSlot, after = 2;
  for (bool ends = false; !ends; ++after) {
    const uint32_t w = uni(code[2u * after]), sub = (w >> 8) & 0xffu;
    ends = (w & VI_ENDS) != 0u;
    if ((w & 0x7fu) != VOP_RED) continue;  // VOP_ENDSWEEP
    const uint32_t how = sub & (0xfu | VRF_SQUARE);
    if ((w >> 24) == 0u) how0 = how;
    else how1 = how;
    if (sub & VRF_PAIR) how1 = VR_SUM | VRF_SQUARE;
  }
  const uint32_t tlog = HDR(team_log2), tx = 1u << tlog, ty = nthreads >> tlog;
  const bool f32 = m.dtype == VDT_F32;
  const uint32_t esz = f32 ? 4u : 2u;
  const uint64_t row_bytes = static_cast<uint64_t>(m.rstride[0]) * esz, step = row_bytes * ty;
  const uint32_t unit[DVM_VEC_MAXR] = {1u, 0u, 0u, 0u};
  const uint32_t n_ridx = HDR(n_ridx), r_chunk = HDR(r_chunk), k_per_chunk = HDR(k_per_chunk), inner_extent = HDR(inner_extent);

  for (uint32_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    const uint32_t k_own = item * tx + (tid & (tx - 1u));
    const uint32_t kidx = k_own < n_kidx ? k_own : n_kidx - 1u;
    // columns this lane starts too late for eight of them
    const uint32_t c = static_cast<uint32_t>(space_offset(kidx, kdims, n_kdim, unit, true));
    const uint32_t late = c + E > inner_extent ? c + E - inner_extent : 0u;
    uint32_t r = 0, r_end = n_ridx;
    if (r_chunk != 0u) {  // a reduce shared between workgroups: the lane's part of the rows
      const uint64_t lo = static_cast<uint64_t>(kidx / k_per_chunk) * r_chunk, hi = lo + r_chunk;
      r = lo < n_ridx ? static_cast<uint32_t>(lo) : n_ridx;
      r_end = hi < n_ridx ? static_cast<uint32_t>(hi) : n_ridx;
    }
    r += tid >> tlog;
    uint64_t at = m.addr + (space_offset(kidx, kdims, n_kdim, m.kstride, true) - late) * esz + static_cast<uint64_t>(r) * row_bytes;
    ColAcc r0, r1;
    FOR_E {
      r0.v[e] = red_identity(how0 & 0xfu);
      r1.v[e] = red_identity(how1 & 0xfu);
    }
    uint32_t left = r < r_end ? (r_end - r + ty - 1u) / ty : 0u;  // rows of this lane
    if (f32) {
      constexpr int NR = 8;
      for (; left >= NR; left -= NR, at += NR * step) col_rows<NR, true, false>(at, step, left, m.dtype, how0, how1, r0, r1);
      if (left != 0u) col_rows<NR, true, true>(at, step, left, m.dtype, how0, how1, r0, r1);
    } else {
      constexpr int NR = 16;
      for (; left >= NR; left -= NR, at += NR * step) col_rows<NR, false, false>(at, step, left, m.dtype, how0, how1, r0, r1);
      if (left != 0u) col_rows<NR, false, true>(at, step, left, m.dtype, how0, how1, r0, r1);
    }
    if (how0 != kNoSlot) col_combine(r0, how0 & 0xfu, tlog, tid, nthreads);
    if (how1 != kNoSlot) col_combine(r1, how1 & 0xfu, tlog, tid, nthreads);
    if (tid >= tx || k_own >= n_kidx) continue;
    float v[E];
    FOR_E v[e] = 0.0f;
    for (uint32_t pc = after;; ++pc) {
      const uint32_t w = uni(code[2u * pc]), imm = uni(code[2u * pc + 1u]);
      const uint32_t op = w & 0x7fu, sub = (w >> 8) & 0xffu, kind = (w >> 16) & 0xfu, rnd = (w >> 20) & 0x3u, a = w >> 24;
      if (op == VOP_END) break;
      if (op == VOP_FIN) {
        FOR_E v[e] = static_cast<float>(a == 0u ? r0.v[e] : r1.v[e]);
      } else if (op == VOP_BINF) {
        FOR_E {
          const float y = kind == VK_IMM ? __uint_as_float(imm) : v[e];
          float x = v[e];
          switch (sub & 0x3fu) {
            case VB_ADD: x = x + y; break;
            case VB_SUB: x = x - y; break;
            case VB_RSUB: x = y - x; break;
            case VB_MUL: x = x * y; break;
            case VB_DIV: x = x / y; break;
            case VB_RDIV: x = y / x; break;
            case VB_MIN: x = x < y ? x : y; break;
            default: x = x > y ? x : y; break;
          }
          v[e] = rnd == VRND_F16 ? round_f16(x) : (rnd == VRND_BF16 ? round_bf16(x) : x);
        }
      } else if (op == VOP_CAST) {
        FOR_E v[e] = rnd == VRND_F16 ? round_f16(v[e]) : (rnd == VRND_BF16 ? round_bf16(v[e]) : v[e]);
      } else {  // VOP_ST
        const VMemDesc o = desc_of(a);
        const uint64_t per = (o.flags & VMF_GATHER) ? o.flags >> 8 : 1u;
        col_store(o, space_offset(kidx, kdims, n_kdim, o.kstride, true) - late * per, v);
      }
    }
  }
#undef HDR
}
