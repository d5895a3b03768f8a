// gfx950 vector VM, row build: programs that reduce the innermost axis and whose rows (the whole reduced space of an
// output) fit the registers of their teams (VS_ROW in isa_gfx950.h) run here.
//
// What bounds such a program (a normalisation, a softmax) is memory, as long as the lanes ask for enough of it at once
// and issue little else. The sweep build walks a row in rounds of two slabs a lane: a row of 4096 elements on one wave is
// four trips to memory one after the other, per sweep, with the decode of every instruction between them, and what a
// second sweep needs again is parked in local memory or fetched again. Here a lane holds UR slabs of eight elements (1
// to 8: UR * team is the row, and only the last slab can be ragged), so a sweep is one round: every load of an operand
// is in flight at once, an instruction is decoded once for the whole row, and the accumulator keeps the row from one
// sweep to the next. The host drops the loads and operations at the head of a sweep whose result the accumulator
// already holds (Compiler::BuildRowCode): a batch of rows is read once, exp(x - max) of a softmax is computed once.
//
// Two things keep the interpreter loop free of per-lane branches and of calls (either makes the compiler save the row
// around it): lanes past the end of a row, and the lane that holds its last few elements, load the row's last eight
// elements instead (`shift` of them belong to other lanes: reduces and stores leave those out), and their stores go
// through a buffer descriptor as long as the row, whose range check drops what they must not write. Rows may start at
// any address their element type allows: the 128-bit accesses need no more than that.
//
// The instruction words are those of the generic interpreter, arranged by the host in a section of the blob of their own
// (at most 64 words: lane i of every wave holds word i and memory operand i's descriptor in registers, and a fetch is
// v_readlane instead of a read of local memory). Each instruction computes what the generic kernel computes, so both
// give the same results but for the order in which the fp64 partials of a reduce are added.
//
// A row may also be the planes of a channel (PLANES; kernels in vm_vector_planes.hip): two reduced axes, rdims[1] planes of
// inner_extent elements, one plane stride for every operand of a sweep. A lane's slabs then lie in planes of their own, and
// each of them may be the ragged last one of its plane. What bounds these programs is the trips to memory of a few workgroups,
// not bandwidth: here a channel is one trip, and every operand's loads of it are in flight at once. Batch-norm in training
// (fp32, sums of x and x^2, us on MI355X) in rounds, which go element by element where a plane does not start on 16 bytes / here:
// [9,427,35,35] 41.7 / 17.1, [17,30,35,35] 38.7 / 13.2, [10,43,14,14] 16.5 / 8.9, [32,512,7,7] 20.1 / 10.3, [5,52,32,32]
// 12.4 / 10.2, [40,2048,27,27] 386 / 163.
#ifndef DVM_DEVICE_VM_VECTOR_ROW_H_
#define DVM_DEVICE_VM_VECTOR_ROW_H_
#include <type_traits>

#include "vec_common.h"

#pragma clang fp contract(off)  // (every instruction rounds its own result, as on the other builds)

namespace {

// the program, copied from the kernel argument once per workgroup
__shared__ __align__(16) uint32_t prog_lds[DVM_PARAM_BYTES / 4];

#define FOR_R _Pragma("unroll") for (int u = 0; u < UR; ++u)
// One slab after the other, as written: the scheduler would otherwise interleave all of a lane's elements through a
// division's or an exponential's dozen instructions, and the temporaries of 64 of those do not fit beside the row.
#define SLAB_DONE() __builtin_amdgcn_sched_barrier(0)

typedef uint32_t vu4_any __attribute__((ext_vector_type(4), aligned(2)));  // 16 bytes at any address of a 16- or 32-bit element

// (single floats and not 8-float vectors: the compiler has to keep a vector in neighbouring registers, and an interpreter
// loop over 8-register tuples ended with 300 registers in scratch memory)
template <int UR>
struct RowAcc {
  float v[UR][E];
};

struct RowDesc {  // a memory operand at the row of the wave; the same in all lanes
  uint64_t addr;
  uint32_t dtype;
};

// Where a lane's slabs lie: element offset of slab 0 (slab u is u * team * 8 further), of the last slab, and how many of
// the last slab's elements belong to other lanes (0: none; 8: all, the lane has no such slab).
struct RowLane {
  static constexpr bool kPlanes = false;
  uint32_t first, last, shift;
  uint32_t step;  // team * 8
  bool wide32;    // every operand of a row is fp32: the lanes of a wave hold its slabs (but the last) in two runs of four elements a lane
  uint32_t row;   // elements of a row
};
// The same for a row of planes: every slab's element offset, and four bits per slab of elements that belong to other lanes.
template <int UR>
struct PlaneLane {
  static constexpr bool kPlanes = true;
  uint32_t off[UR];
  uint32_t shifts;
  uint32_t row;  // elements from the first of the first plane to behind the last of the last
};

// A per-lane value as it is now: what is computed from it stays where it stands instead of being hoisted out of the
// interpreter loop (masks and offsets of every slab would occupy registers for the whole launch).
__device__ __forceinline__ uint32_t fresh_v(uint32_t x) {
  asm volatile("" : "+v"(x));
  return x;
}

__device__ __forceinline__ void widen_bf16(vu4 a, float (&r)[E]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    r[2 * i] = __uint_as_float(a[i] << 16);
    r[2 * i + 1] = __uint_as_float(a[i] & 0xffff0000u);
  }
}
__device__ __forceinline__ void widen_f16(vu4 a, float (&r)[E]) {
  const vh8 h = __builtin_bit_cast(vh8, a);
  FOR_E r[e] = static_cast<float>(h[e]);
}
__device__ __forceinline__ void join32(vu4 a, vu4 b, float (&r)[E]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    r[i] = __uint_as_float(a[i]);
    r[4 + i] = __uint_as_float(b[i]);
  }
}
__device__ __forceinline__ vu4 load16(uint64_t base, uint32_t off) {  // base in scalar registers, the lane's offset in one vector register
  return *reinterpret_cast<const DVM_GLOBAL vu4_any *>(reinterpret_cast<const DVM_GLOBAL char *>(base) + off);
}
__device__ __forceinline__ void store16(uint64_t base, uint32_t off, vu4 v) {
  *reinterpret_cast<DVM_GLOBAL vu4_any *>(reinterpret_cast<DVM_GLOBAL char *>(base) + off) = v;
}

// Where a lane's 32-bit slabs before the last lie, in bytes: their first half, and from there to the second. With both halves of
// eight elements side by side an access instruction of a wave touches half of every 32 bytes of 2 KB, and each of the two
// moves all of its lines. (A program with 16-bit rows as well keeps its elements where those have them.) Side by side / in
// runs, us on MI355X: RMSNorm fp32 [2048,32001] 132.1 / 122.6, [8192,4095] 63.6 / 59.5, [3000,11000] 62.5 / 55.6, [4096,2048]
// 16.0 / 14.9; softmax fp32 [2048,32000] 149.8 / 145.6, [2048,32001] 150.5 / 149.7, [2048,8192] 38.5 / 37.1.
__device__ __forceinline__ uint32_t first32(const RowLane &l) {
  const uint32_t first = fresh_v(l.first);
  return l.wide32 ? ((first & ~511u) << 2) + ((first & 511u) << 1) : first << 2;
}
__device__ __forceinline__ uint32_t half32(const RowLane &l) { return l.wide32 ? 1024u : 16u; }

// The row of an operand as it lies in memory: 32-bit elements take both halves, 16-bit ones the first.
template <int UR>
struct RowRaw {
  vu4 a[UR], b[UR];
};
template <int UR, typename L>
__device__ __forceinline__ void row_fetch32(const RowDesc &d, const L &l, RowRaw<UR> &r) {
  if constexpr (L::kPlanes) {
    FOR_R {
      const uint32_t off = fresh_v(l.off[u]) * 4u;
      r.a[u] = load16(d.addr, off);
      r.b[u] = load16(d.addr + 16, off);
    }
    return;
  } else {
  const uint32_t first = first32(l), last = fresh_v(l.last) * 4u, step = l.step * 4u, half = half32(l);
  FOR_R {
    const uint64_t base = d.addr + (u < UR - 1 ? u * step : 0u);
    const uint32_t off = u < UR - 1 ? first : last;
    r.a[u] = load16(base, off);
    r.b[u] = load16(base + (u < UR - 1 ? half : 16u), off);
  }
  }
}
template <int UR, typename L>
__device__ __forceinline__ void row_fetch16(const RowDesc &d, const L &l, vu4 (&a)[UR]) {
  if constexpr (L::kPlanes) {
    FOR_R a[u] = load16(d.addr, fresh_v(l.off[u]) * 2u);
    return;
  } else {
  const uint32_t first = fresh_v(l.first) * 2u, last = fresh_v(l.last) * 2u, step = l.step * 2u;
  FOR_R a[u] = load16(d.addr + (u < UR - 1 ? u * step : 0u), u < UR - 1 ? first : last);
  }
}
template <int UR>
__device__ __forceinline__ void row_widen(uint32_t dtype, const vu4 (&a)[UR], RowAcc<UR> &out) {
  if (dtype == VDT_BF16) {
    FOR_R widen_bf16(a[u], out.v[u]);
  } else {
    FOR_R widen_f16(a[u], out.v[u]);
  }
}

template <int UR, typename L>
__device__ __forceinline__ void row_load(const RowDesc &d, const L &l, RowAcc<UR> &out) {
  if (d.dtype == VDT_F32) {
    RowRaw<UR> r;
    row_fetch32<UR>(d, l, r);
    FOR_R join32(r.a[u], r.b[u], out.v[u]);
  } else {
    vu4 a[UR];
    row_fetch16<UR>(d, l, a);
    row_widen<UR>(d.dtype, a, out);
  }
}

// The last slab's elements one by one, through a descriptor of the row: what lies past its end is dropped.
__device__ __forceinline__ void store_ragged32(const RowDesc &d, uint32_t row, uint32_t at, uint32_t shift, const float (&v)[E]) {
  const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(d.addr), 0, static_cast<int>(row * 4u), 0x00027000);
  FOR_E __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[e]), rsrc, static_cast<uint32_t>(e) >= shift ? at * 4u + 4u * e : 0xfffffff0u, 0, 0);
}
__device__ __forceinline__ void store_ragged16(const RowDesc &d, uint32_t row, uint32_t at, uint32_t shift, vu4 v) {
  const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(d.addr), 0, static_cast<int>(row * 2u), 0x00027000);
  FOR_E __builtin_amdgcn_raw_buffer_store_b16(static_cast<uint16_t>(v[e >> 1] >> (16 * (e & 1))), rsrc,
                                                  static_cast<uint32_t>(e) >= shift ? at * 2u + 2u * e : 0xfffffff0u, 0, 0);
}
__device__ __forceinline__ vu4 slab16(uint32_t dtype, const float (&v)[E]) {
  vu4 a;
  if (dtype == VDT_BF16) {
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = pack_bf16(v[2 * i], v[2 * i + 1]);
  } else {
    vh8 h;
    FOR_E h[e] = static_cast<_Float16>(v[e]);
    a = __builtin_bit_cast(vu4, h);
  }
  return a;
}
// A row of planes: the whole slabs of a wave with 128-bit stores (through the descriptor as well, which drops those that are
// not whole), the ragged ones, where the wave has any, element by element.
template <int UR>
__device__ __forceinline__ void row_store(const RowDesc &d, const PlaneLane<UR> &l, const RowAcc<UR> &in) {
  const uint32_t isz = d.dtype == VDT_F32 ? 4u : 2u;
  const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(d.addr), 0, static_cast<int>(l.row * isz), 0x00027000);
  FOR_R {
    const uint32_t shift = (fresh_v(l.shifts) >> (4 * u)) & 15u, off = fresh_v(l.off[u]);
    const uint32_t at = shift == 0u ? off * isz : 0xffffff00u;
    if (d.dtype == VDT_F32) {
      const vf4 lo = {in.v[u][0], in.v[u][1], in.v[u][2], in.v[u][3]}, hi = {in.v[u][4], in.v[u][5], in.v[u][6], in.v[u][7]};
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(vu4, lo), rsrc, at, 0, 0);
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(vu4, hi), rsrc, at + 16u, 0, 0);
      if (!wave_all(shift == 0u || shift == 8u)) store_ragged32(d, l.row, off, shift == 0u ? 8u : shift, in.v[u]);
    } else {
      const vu4 a = slab16(d.dtype, in.v[u]);
      __builtin_amdgcn_raw_buffer_store_b128(a, rsrc, at, 0, 0);
      if (!wave_all(shift == 0u || shift == 8u)) store_ragged16(d, l.row, off, shift == 0u ? 8u : shift, a);
    }
    SLAB_DONE();
  }
}
template <int UR>
__device__ __forceinline__ void row_store(const RowDesc &d, const RowLane &l, const RowAcc<UR> &in) {
  const bool whole = wave_all(fresh_v(l.shift) == 0u);
  const uint32_t isz = d.dtype == VDT_F32 ? 4u : 2u;
  const uint32_t last = fresh_v(l.last) * isz, step = l.step * isz;
  if (d.dtype == VDT_F32) {
    const uint32_t first = first32(l), half = half32(l);
    FOR_R {
      const uint64_t base = d.addr + (u < UR - 1 ? u * step : 0u);
      if (u == UR - 1 && !whole) {
        store_ragged32(d, l.row, l.last, fresh_v(l.shift), in.v[u]);
      } else {
        const vf4 lo = {in.v[u][0], in.v[u][1], in.v[u][2], in.v[u][3]}, hi = {in.v[u][4], in.v[u][5], in.v[u][6], in.v[u][7]};
        store16(base, u < UR - 1 ? first : last, __builtin_bit_cast(vu4, lo));
        store16(base + (u < UR - 1 ? half : 16u), u < UR - 1 ? first : last, __builtin_bit_cast(vu4, hi));
      }
    }
    return;
  }
  const uint32_t first = fresh_v(l.first) * isz;
  FOR_R {
    const vu4 a = slab16(d.dtype, in.v[u]);
    if (u == UR - 1 && !whole) {
      store_ragged16(d, l.row, l.last, fresh_v(l.shift), a);
    } else {
      store16(d.addr + (u < UR - 1 ? u * step : 0u), u < UR - 1 ? first : last, a);
    }
    SLAB_DONE();
  }
}

template <int UR>
__device__ __forceinline__ void row_round(RowAcc<UR> &a, uint32_t rnd) {
  if (rnd == VRND_NONE) return;
  if (rnd == VRND_F16) {
    FOR_R FOR_E a.v[u][e] = round_f16(a.v[u][e]);
  } else {
    FOR_R FOR_E a.v[u][e] = round_bf16(a.v[u][e]);
  }
}
__device__ __forceinline__ float round_one(float x, uint32_t rnd) { return rnd == VRND_F16 ? round_f16(x) : (rnd == VRND_BF16 ? round_bf16(x) : x); }

// acc = acc (sub) s with one value s per lane
template <int UR>
__device__ __forceinline__ void row_lane_binary(RowAcc<UR> &acc, uint32_t sub, float s) {
  switch (sub) {
    case VB_ADD: FOR_R FOR_E acc.v[u][e] = acc.v[u][e] + s; break;
    case VB_SUB: FOR_R FOR_E acc.v[u][e] = acc.v[u][e] - s; break;
    case VB_RSUB: FOR_R FOR_E acc.v[u][e] = s - acc.v[u][e]; break;
    case VB_MUL: FOR_R FOR_E acc.v[u][e] = acc.v[u][e] * s; break;
    case VB_DIV: FOR_R { FOR_E acc.v[u][e] = acc.v[u][e] / s; SLAB_DONE(); } break;
    case VB_RDIV: FOR_R { FOR_E acc.v[u][e] = s / acc.v[u][e]; SLAB_DONE(); } break;
    case VB_MIN: FOR_R FOR_E acc.v[u][e] = acc.v[u][e] < s ? acc.v[u][e] : s; break;
    default: FOR_R FOR_E acc.v[u][e] = acc.v[u][e] > s ? acc.v[u][e] : s; break;  // VB_MAX
  }
}
// acc = acc (sub) operand, element by element (on NaN the second operand of min / max wins, as in the reference functors,
// src/vm_gpu.cu:222-233). The operand is read from its raw form as it is used: widened into an array of its own first,
// it would need another 8 * UR registers. GET(u, e): element e of slab u.
template <int UR, typename GET>
__device__ __forceinline__ void row_binary(RowAcc<UR> &acc, uint32_t sub, GET get) {
  switch (sub) {
    case VB_ADD: FOR_R FOR_E acc.v[u][e] = acc.v[u][e] + get(u, e); break;
    case VB_SUB: FOR_R FOR_E acc.v[u][e] = acc.v[u][e] - get(u, e); break;
    case VB_RSUB: FOR_R FOR_E acc.v[u][e] = get(u, e) - acc.v[u][e]; break;
    case VB_MUL: FOR_R FOR_E acc.v[u][e] = acc.v[u][e] * get(u, e); break;
    case VB_DIV: FOR_R { FOR_E acc.v[u][e] = acc.v[u][e] / get(u, e); SLAB_DONE(); } break;
    case VB_RDIV: FOR_R { FOR_E acc.v[u][e] = get(u, e) / acc.v[u][e]; SLAB_DONE(); } break;
    case VB_MIN: FOR_R FOR_E { const float y = get(u, e); acc.v[u][e] = acc.v[u][e] < y ? acc.v[u][e] : y; } break;
    default: FOR_R FOR_E { const float y = get(u, e); acc.v[u][e] = acc.v[u][e] > y ? acc.v[u][e] : y; } break;
  }
}
__device__ __forceinline__ float bf16_at(const vu4 &a, int e) { return __uint_as_float((e & 1) ? (a[e >> 1] & 0xffff0000u) : (a[e >> 1] << 16)); }
__device__ __forceinline__ float f16_at(const vu4 &a, int e) { return static_cast<float>(__builtin_bit_cast(vh8, a)[e]); }
template <int UR>
__device__ __forceinline__ void row_binary16(RowAcc<UR> &acc, uint32_t sub, uint32_t dtype, const vu4 (&a)[UR]) {
  if (dtype == VDT_BF16) {
    row_binary<UR>(acc, sub, [&](int u, int e) { return bf16_at(a[u], e); });
  } else {
    row_binary<UR>(acc, sub, [&](int u, int e) { return f16_at(a[u], e); });
  }
}

// What a reduce adds to a lane's partial: the eight elements of a slab pairwise in fp32, slabs in fp64 (the generic
// kernel's order inside a lane). SQUARE: of the squares. The accumulator itself stays as it is.
template <int UR, bool SQUARE, typename L>
__device__ __forceinline__ double row_sum(const RowAcc<UR> &x, const L &l) {
  uint32_t shift = 0;
  if constexpr (!L::kPlanes) shift = fresh_v(l.shift);
  double r = 0.0;
  FOR_R {
    float d[E];
    FOR_E d[e] = SQUARE ? x.v[u][e] * x.v[u][e] : x.v[u][e];
    if constexpr (L::kPlanes) shift = (fresh_v(l.shifts) >> (4 * u)) & 15u;
    if (L::kPlanes || u == UR - 1) FOR_E d[e] = static_cast<uint32_t>(e) >= shift ? d[e] : 0.0f;
#pragma unroll
    for (int w = 1; w < E; w <<= 1)
#pragma unroll
      for (int e = 0; e + w < E; e += 2 * w) d[e] = d[e] + d[e + w];
    r += static_cast<double>(d[0]);
    SLAB_DONE();
  }
  return r;
}
// max / min round nothing, so the slabs combine in fp32 (v_maximum3_f32: NaN propagates, as NumPy's max / min)
template <int UR, bool MAX, typename L>
__device__ __forceinline__ double row_extreme(const RowAcc<UR> &x, const L &l) {
  constexpr float idv = MAX ? -__builtin_huge_valf() : __builtin_huge_valf();
  uint32_t shift = 0;
  if constexpr (!L::kPlanes) shift = fresh_v(l.shift);
  float m = idv;
  FOR_R {
    float d[E];
    FOR_E d[e] = x.v[u][e];
    if constexpr (L::kPlanes) shift = (fresh_v(l.shifts) >> (4 * u)) & 15u;
    if (L::kPlanes || u == UR - 1) FOR_E d[e] = static_cast<uint32_t>(e) >= shift ? d[e] : idv;
    FOR_E m = MAX ? __builtin_elementwise_maximum(m, d[e]) : __builtin_elementwise_minimum(m, d[e]);
    SLAB_DONE();
  }
  return static_cast<double>(m);
}

// Arithmetic on one value per lane between the sweeps.
__device__ __forceinline__ float row_one_binary(uint32_t op, uint32_t sub, float x, float y) {
  if (op == VOP_BINF) {
    switch (sub & 0x3fu) {
      case VB_ADD: return x + y;
      case VB_SUB: return x - y;
      case VB_RSUB: return y - x;
      case VB_MUL: return x * y;
      case VB_DIV: return x / y;
      case VB_RDIV: return y / x;
      case VB_MIN: return x < y ? x : y;
      default: return x > y ? x : y;
    }
  }
  const uint32_t t = sub & 0x7u;  // VOP_CMP
  const bool c = t == VCMP_EQ ? x == y : t == VCMP_NE ? x != y : t == VCMP_GT ? x > y : t == VCMP_GE ? x >= y : t == VCMP_LT ? x < y : x <= y;
  return c ? 1.0f : 0.0f;
}
__device__ __forceinline__ float row_one_unary(uint32_t sub, float x) {
  switch (sub) {
    case VU_SQRT: return sqrtf(x);
    case VU_LOG: return logf(x);
    case VU_ABS: return fabsf(x);
    case VU_EXP: return exp_f32(x);
    case VU_ISFINITE: return isfinite(x) ? 1.0f : 0.0f;
    case VU_ROUND: return rintf(x);
    case VU_FLOOR: return floorf(x);
    case VU_CEIL: return ceilf(x);
    default: return truncf(x);
  }
}

template <int UR, bool PLANES>
__device__ __forceinline__ void vm_vector_row(const VmParam &p) {
  // (Four slabs are faster this way: residual RMSNorm bf16 [4490,1648] 14.8 us, 16.7 the other; over 172 softmaxes and residual
  // norms of 300 to 8192 rows the other way is 2.7 % slower on average, 13 % at most, and 4 % faster at 300 x 13000.)
  if constexpr (UR == 4) {
    const uint32_t rc = reinterpret_cast<const VVecHeader *>(p.w)->row_code;
    fetch_used_words(prog_lds, p.w, ((rc & 0xffffu) + (rc >> 16)) * 2);
  } else {
    fetch_program(prog_lds, p.w, [&]() {
      const uint32_t rc = prog_lds[offsetof(VVecHeader, row_code) / 4];
      return ((rc & 0xffffu) + (rc >> 16)) * 2;
    });
  }
  auto word32 = [&](uint32_t i) -> uint32_t { return uni(prog_lds[i]); };
#define HDR(field) word32(static_cast<uint32_t>(offsetof(VVecHeader, field) / 4))
  const uint32_t tid = threadIdx.x, lane = tid & 63u, nthreads = blockDim.x;
  // lane i holds instruction word i and the fields of memory operand i
  bool other_row;  // operand `lane` varies along the row and is not fp32
  uint32_t code_lo, code_hi, m_addr_lo, m_addr_hi, m_type, m_ks0, m_ks1;
  {
    const uint32_t row_code = HDR(row_code), off = row_code & 0xffffu, n = row_code >> 16;
    const uint32_t i = off + (lane < n ? lane : n - 1u);
    code_lo = prog_lds[2u * i];
    code_hi = prog_lds[2u * i + 1u];
    const uint32_t n_mem = HDR(n_mem), j = lane < n_mem ? lane : n_mem - 1u;
    const vu4 *dq = reinterpret_cast<const vu4 *>(prog_lds + 2u * (HDR(mem_off) + j * static_cast<uint32_t>(sizeof(VMemDesc) / 8)));
    const vu4 q0 = dq[0], q1 = dq[1];
    m_addr_lo = q0[0];
    m_addr_hi = q0[1];
    m_type = q0[2];
    other_row = m_type != VDT_F32 && (q0[3] & VMF_VEC) != 0;
    m_ks0 = q1[0];
    m_ks1 = q1[1];
  }
  const uint32_t n_kidx = HDR(n_kidx), n_kdim = HDR(n_kdim), n_items = HDR(n_items);
  const uint32_t kd_extent = HDR(kdims[0].extent), kd_magic = HDR(kdims[0].magic), kd_shift = HDR(kdims[0].shift);
  const bool team_is_block = HDR(team_is_block) != 0u;  // (else one wave per row)
  const uint32_t wave = uni(tid >> 6);
  typename std::conditional<PLANES, PlaneLane<UR>, RowLane>::type rl;
  if constexpr (PLANES) {
    const uint32_t team = team_is_block ? nthreads : 64u, at = team_is_block ? tid : lane;
    const uint32_t groups = HDR(rdims[0].extent), magic = HDR(rdims[0].magic), dshift = HDR(rdims[0].shift), n_ridx = HDR(n_ridx);
    const uint32_t plane_elems = HDR(inner_extent), plane_stride = HDR(plane_stride);
    rl.row = (HDR(rdims[1].extent) - 1u) * plane_stride + plane_elems;
    rl.shifts = 0;
    FOR_R {
      const uint32_t i = at + static_cast<uint32_t>(u) * team, g = i < n_ridx ? i : n_ridx - 1u;
      const uint32_t plane = (__umulhi(g, magic) + g) >> dshift, c = (g - plane * groups) * E, end = plane_elems - E;
      rl.off[u] = plane * plane_stride + (c < end ? c : end);
      const uint32_t shift = i >= n_ridx ? static_cast<uint32_t>(E) : (c <= end ? 0u : c - end);
      rl.shifts |= shift << (4 * u);
    }
  } else {
    const uint32_t team = team_is_block ? nthreads : 64u, at = team_is_block ? tid : lane;
    rl.row = HDR(inner_extent);
    rl.step = team * E;
    rl.first = at * E;
    rl.wide32 = __ballot(other_row) == 0;
    const uint32_t c = (at + (UR - 1) * team) * E, end = rl.row - E;
    rl.last = c < end ? c : end;
    rl.shift = c <= end ? 0u : (c - end < E ? c - end : static_cast<uint32_t>(E));
  }
  vf4 *planes = reinterpret_cast<vf4 *>(lds + nthreads);  // V registers (at most two slabs a lane)

  SRegs sr;
  sr.s0 = sr.s1 = sr.s2 = sr.s3 = sr.s4 = sr.s5 = sr.s6 = sr.s7 = 0.0f;
  RowAcc<UR> acc;
  FOR_R FOR_E acc.v[u][e] = 0.0f;
  float x = 0.0f;  // the accumulator between sweeps: one value per lane
  double racc0 = 0.0, racc1 = 0.0;
  uint32_t red_flip = 0;

  for (uint32_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    const uint32_t kidx = team_is_block ? item : item * (nthreads >> 6) + wave;
    if (kidx >= n_kidx) break;  // (waves with rows of their own: no barrier is skipped)
    uint32_t kc0 = kidx, kc1 = 0;
    if (n_kdim > 1u) {
      kc1 = (static_cast<uint32_t>((static_cast<uint64_t>(kidx) * kd_magic) >> 32) + kidx) >> kd_shift;
      kc0 = kidx - kc1 * kd_extent;
    }
    auto desc_at = [&](uint32_t i) -> RowDesc {
      RowDesc d;
      const uint64_t base = static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readlane(m_addr_lo, i))) |
                            (static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readlane(m_addr_hi, i))) << 32);
      d.dtype = __builtin_amdgcn_readlane(m_type, i);
      const uint64_t k = static_cast<uint64_t>(kc0) * static_cast<uint32_t>(__builtin_amdgcn_readlane(m_ks0, i)) +
                         static_cast<uint64_t>(kc1) * static_cast<uint32_t>(__builtin_amdgcn_readlane(m_ks1, i));
      d.addr = base + k * (d.dtype == VDT_F32 ? 4u : 2u);
      return d;
    };

    bool xmask = false;  // the predicate of VOP_MSK between sweeps
    uint32_t pc = 0;
    while (true) {
      uint32_t w0 = __builtin_amdgcn_readlane(code_lo, pc);
      uint32_t imm = __builtin_amdgcn_readlane(code_hi, pc);
      ++pc;
      uint32_t op = w0 & 0x7fu;
      if (op == VOP_END) break;
      if (op != VOP_SWEEP) {
        // ---- one value per lane ----
        const uint32_t sub = (w0 >> 8) & 0xffu, a = w0 >> 24, kind = (w0 >> 16) & 0xfu, rnd = (w0 >> 20) & 0x3u;
        if (op >= VOP_SRC_BASE) {
          float sv;
          if (kind == VK_MEM) {
            const RowDesc m = desc_at(a);
            sv = elem_load(m.addr, m.dtype, 0);
          } else {
            sv = kind == VK_IMM ? __uint_as_float(imm) : (kind == VK_ACC ? x : sreg_read(sr, a));
          }
          if (op == VOP_LD) {
            x = sv;
          } else if (op == VOP_MSK) {
            xmask = (__float_as_uint(sv) << 1) != 0u;
          } else if (op == VOP_MOVM) {
            x = xmask ? sv : x;
          } else {
            x = row_one_binary(op, sub, x, sv);
            if (op == VOP_BINF) {
              x = round_one(x, rnd);
              if (kind == VK_SREG2) {
                x = row_one_binary(VOP_BINF, imm & 0x3fu, x, sreg_read(sr, (imm >> 8) & 0xffu));
                x = round_one(x, (imm >> 16) & 0x3u);
              }
            }
          }
          continue;
        }
        switch (op) {
          case VOP_FIN: x = static_cast<float>(a == 0 ? racc0 : racc1); break;
          case VOP_LDS: x = sreg_read(sr, a); break;
          case VOP_LDI: x = __uint_as_float(imm); break;
          case VOP_STS: sreg_write(sr, a, x); break;
          case VOP_UN: x = round_one(row_one_unary(sub, x), rnd); break;
          case VOP_CAST: x = round_one(x, rnd); break;  // VC_RND
          default: {                                    // VOP_ST: one value per row (any lane's: the first one writes)
            const RowDesc m = desc_at(a);
            const uint32_t none = fresh_v((team_is_block ? tid : lane) == 0u ? 0u : static_cast<uint32_t>(E));
            const float out[E] = {x, x, x, x, x, x, x, x};
            if (m.dtype == VDT_F32) {
              store_ragged32(m, 1u, 0u, none, out);
            } else {
              const uint32_t h = m.dtype == VDT_BF16 ? f32_to_bf16_bits(x) : __builtin_bit_cast(uint16_t, static_cast<_Float16>(x));
              store_ragged16(m, 1u, 0u, none, vu4{h, 0u, 0u, 0u});
            }
            break;
          }
        }
        continue;
      }

      // ---- a sweep: one round ----
      const uint32_t k0 = imm & 0xfu, k1 = (imm >> 4) & 0xfu;
      racc0 = racc1 = 0.0;
      bool ends;
      do {
        w0 = __builtin_amdgcn_readlane(code_lo, pc);
        imm = __builtin_amdgcn_readlane(code_hi, pc);
        ++pc;
        op = w0 & 0x7fu;
        ends = (w0 & VI_ENDS) != 0;
        const uint32_t sub = (w0 >> 8) & 0xffu, rnd = (w0 >> 20) & 0x3u, a = w0 >> 24, kind = (w0 >> 16) & 0xfu;
        switch (op) {
          case VOP_LD: {
            const RowDesc d = desc_at(a);
            if ((w0 & VI_LD_PAIR) != 0) {  // 16-bit rows of one type: the next instruction's operand in the same trip
              w0 = __builtin_amdgcn_readlane(code_lo, pc);
              ++pc;
              ends = (w0 & VI_ENDS) != 0;
              const RowDesc d2 = desc_at(w0 >> 24);
              vu4 ra[UR], rb[UR];
              row_fetch16<UR>(d, rl, ra);
              row_fetch16<UR>(d2, rl, rb);
              row_widen<UR>(d.dtype, ra, acc);
              row_binary16<UR>(acc, (w0 >> 8) & 0x3fu, d.dtype, rb);
              row_round<UR>(acc, (w0 >> 20) & 0x3u);
            } else {
              row_load<UR>(d, rl, acc);
            }
            break;
          }
          case VOP_BINF: {
            if (kind == VK_MEM) {
              const RowDesc d = desc_at(a);
              auto pre = [&]() {  // an S-register binary in front, while the operand is on its way
                if (imm & VI_PRE_SREG) {
                  row_lane_binary<UR>(acc, imm & 0x3fu, sreg_read(sr, (imm >> 8) & 0xffu));
                  row_round<UR>(acc, (imm >> 16) & 0x3u);
                }
              };
              if (d.dtype == VDT_F32) {
                RowRaw<UR> r;
                row_fetch32<UR>(d, rl, r);
                pre();
                row_binary<UR>(acc, sub & 0x3fu, [&](int u, int e) { return __uint_as_float(e < 4 ? r.a[u][e] : r.b[u][e - 4]); });
              } else {
                vu4 r[UR];
                row_fetch16<UR>(d, rl, r);
                pre();
                row_binary16<UR>(acc, sub & 0x3fu, d.dtype, r);
              }
              row_round<UR>(acc, rnd);
            } else if (kind == VK_ACC) {
              row_binary<UR>(acc, sub & 0x3fu, [&](int u, int e) { return acc.v[u][e]; });
              row_round<UR>(acc, rnd);
            } else if (kind == VK_REG) {
              if constexpr (UR <= U) {
                Acc t;
                vreg_load(planes, a, sub >> 6, nthreads, tid, t);
                row_binary<UR>(acc, sub & 0x3fu, [&](int u, int e) { return t.v[u][e]; });
                row_round<UR>(acc, rnd);
              }
            } else {
              row_lane_binary<UR>(acc, sub & 0x3fu, kind == VK_IMM ? __uint_as_float(imm) : sreg_read(sr, a));
              row_round<UR>(acc, rnd);
              if (kind == VK_SREG2) {
                row_lane_binary<UR>(acc, imm & 0x3fu, sreg_read(sr, (imm >> 8) & 0xffu));
                row_round<UR>(acc, (imm >> 16) & 0x3u);
              }
            }
            break;
          }
          case VOP_RED: {
            const uint32_t rk = sub & 0xfu;
            double t;
            if (rk == VR_SUM) {
              t = (sub & VRF_SQUARE) ? row_sum<UR, true>(acc, rl) : row_sum<UR, false>(acc, rl);
              if (sub & VRF_PAIR) racc1 = row_sum<UR, true>(acc, rl);
            } else {
              t = rk == VR_MAX ? row_extreme<UR, true>(acc, rl) : row_extreme<UR, false>(acc, rl);
            }
            if (a == 0u) {
              racc0 = t;
            } else {
              racc1 = t;
            }
            break;
          }
          case VOP_ST: {
            const RowDesc d = desc_at(a);
            row_store<UR>(d, rl, acc);
            break;
          }
          case VOP_LDS: {
            const float v = sreg_read(sr, a);
            FOR_R FOR_E acc.v[u][e] = v;
            break;
          }
          case VOP_LDI: FOR_R FOR_E acc.v[u][e] = __uint_as_float(imm); break;
          case VOP_SPLAT: FOR_R FOR_E acc.v[u][e] = x; break;
          case VOP_LDR:
            if constexpr (UR <= U) {
              Acc t;
              vreg_load(planes, a, sub, nthreads, tid, t);
              FOR_R FOR_E acc.v[u][e] = t.v[u][e];
            }
            break;
          case VOP_STR:
            if constexpr (UR <= U) {
              Acc t;
              FOR_U t.v[u] = 0.0f;
              FOR_R FOR_E t.v[u][e] = acc.v[u][e];
              vreg_store(planes, a, sub, nthreads, tid, t);
            }
            break;
          case VOP_UN: {
            if (sub == VU_EXP) {
              FOR_R { FOR_E acc.v[u][e] = exp_f32(acc.v[u][e]); SLAB_DONE(); }
            } else {  // VU_ABS
              FOR_R FOR_E acc.v[u][e] = fabsf(acc.v[u][e]);
            }
            row_round<UR>(acc, rnd);
            break;
          }
          case VOP_CAST: row_round<UR>(acc, rnd); break;  // VC_RND
          default: break;                                 // VOP_ENDSWEEP
        }
      } while (!ends);
      x = acc.v[0][0];
      if (k0 <= VR_MIN || k1 <= VR_MIN) red_finish_x(racc0, racc1, k0, k1, 6u, team_is_block, tid, nthreads, red_flip, lds);
    }
  }
#undef HDR
}

}  // namespace

#endif  // DVM_DEVICE_VM_VECTOR_ROW_H_
