// The fused attention launch.
#include <algorithm>
#include <cstdlib>
#include <cmath>
#include <cstddef>
#include <cstring>
#include <stdexcept>

#include "../../../include/dvm_hip.h"
#include "compiler.h"

namespace dvm {

void Compiler::CompileAttn(int gi) {
  const AttnGroup &g = attn_groups_[gi];
  const int r = g.q->rank();
  VAttnHeader h;
  std::memset(&h, 0, sizeof(h));
  h.entry = VE_ATTN;
  h.dtype = MemDType(g.m2->type_id_);
  int64_t nb = 1;
  for (int d = 0; d < r - 2; ++d) nb *= g.q->dim(d);
  h.nb = static_cast<uint32_t>(nb);
  h.sq = static_cast<uint32_t>(g.q->dim(r - 2));
  h.skv = static_cast<uint32_t>(g.k->dim(r - 2));
  h.d = static_cast<uint32_t>(g.q->dim(r - 1));
  h.scale = g.scale;
  h.q_blocks = (h.sq + DVM_ATTN_BQ - 1) / DVM_ATTN_BQ;
  // where the (batch, head) pairs of each operand lie (views are walked in place)
  AttnLayout lay[3] = {AttnOperandLayout(g.q), AttnOperandLayout(g.k), AttnOperandLayout(g.v)};
  uint32_t nb_inner = 1;
  for (const AttnLayout &l : lay) {
    if (!l.ok) Fail("attention operand layout");
    if (l.nb_inner != 1) nb_inner = l.nb_inner;
  }
  if (g.out_store != nullptr && g.out_nb_inner != 1) nb_inner = g.out_nb_inner;
  h.nb_inner = nb_inner;
  for (int i = 0; i < 3; ++i) {
    const NDObject *t = i == 0 ? g.q : (i == 1 ? g.k : g.v);
    h.row_stride[i] = lay[i].row;
    if (lay[i].nb_inner == 1 && nb_inner != 1) {  // dense beside a view with two batch axes: split its batch stride
      const int64_t per = t->dim(r - 2) * t->dim(r - 1);
      h.inner_stride[i] = static_cast<uint32_t>(per);
      h.outer_stride[i] = static_cast<uint32_t>(per * nb_inner);
    } else {
      h.outer_stride[i] = lay[i].outer;
      h.inner_stride[i] = lay[i].inner;
    }
  }
  // the result is dense, [nb][sq][d], unless it goes into a Store through strides
  h.row_stride[3] = h.d;
  h.inner_stride[3] = nb_inner != 1 ? h.sq * h.d : 0;
  h.outer_stride[3] = h.sq * h.d * nb_inner;
  if (g.out_store != nullptr) {
    h.row_stride[3] = g.out_row;
    if (g.out_nb_inner == 1 && nb_inner != 1) {  // one batch stride beside operands with two: split it
      h.inner_stride[3] = g.out_outer;
      h.outer_stride[3] = g.out_outer * nb_inner;
    } else {
      h.inner_stride[3] = g.out_inner;
      h.outer_stride[3] = g.out_outer;
    }
  }
  if (static_cast<uint64_t>(h.nb) * h.q_blocks >= (1ull << 31)) Fail("too many attention blocks");
  std::memset(&prog_->blob, 0, sizeof(VmParam));
  std::memcpy(prog_->blob.w, &h, sizeof(h));
  auto patch = [&](size_t byte_off, int op_id, int ws_slot, int64_t elem_offset = 0) {
    Program::Patch p;
    p.word = static_cast<uint32_t>(byte_off / 8);
    p.op_id = op_id;
    p.ws_slot = ws_slot;
    p.byte_offset = elem_offset * 2;
    p.role = Program::kPatchAligned16;
    prog_->patches.push_back(p);
  };
  patch(offsetof(VAttnHeader, q_addr), lay[0].root->id, -1, lay[0].base);
  patch(offsetof(VAttnHeader, k_addr), lay[1].root->id, -1, lay[1].base);
  patch(offsetof(VAttnHeader, v_addr), lay[2].root->id, -1, lay[2].base);
  // the result goes to the user's store when there is one in this sub-kernel, else to workspace
  const int m2 = g.m2->id;
  if (g.out_store != nullptr) {
    patch(offsetof(VAttnHeader, o_addr), g.out_store->id, -1, g.out_base);
  } else if (store_of_[m2] >= 0 && area_[store_of_[m2]] == area_[m2]) {
    patch(offsetof(VAttnHeader, o_addr), store_of_[m2], -1);
  } else if (ws_slot_[m2] >= 0) {
    patch(offsetof(VAttnHeader, o_addr), -1, ws_slot_[m2]);
  } else {
    Fail("attention result has no destination");
  }
  // eight waves of 32 queries (two per SIMD: one wave's softmax runs under the other's MFMAs) measured 767-788 us
  // on fp16 [8,32,2048,128] against 920-940 us for four waves of 64 queries; DVM_ATTN_WAVES=4 selects the latter
  prog_->threads = 512;
  if (k_->tuning_.attn_waves == 4) prog_->threads = 256;
  prog_->lds_bytes = DVM_ATTN_LDS_BYTES_D(h.d);
  prog_->grid = h.nb * h.q_blocks;
  DivideKeys();
}

constexpr size_t kPartBytes = 8u << 20;

// Hands an attention to the kernel whose waves divide the keys, where that is the faster one.
void Compiler::DivideKeys() {
  VAttnHeader *h = reinterpret_cast<VAttnHeader *>(prog_->blob.w);
  const int forced = k_->tuning_.attn_keys;
  if (forced == 0 || (forced < 0 && k_->tuning_.attn_waves >= 0)) return;
  const uint64_t cus = g_system.core_num > 0 ? g_system.core_num : 256;
  const uint64_t slots = h->d == DVM_ATTN_D ? cus : 2 * cus;  // 128 KB of local memory a workgroup, or 64
  const uint32_t q_blocks = (h->sq - 1) / DVM_ATTN_KEYS_BQ + 1, blocks = (h->skv - 1) / DVM_ATTN_KEYS_BKV + 1;
  const uint64_t tiles = static_cast<uint64_t>(h->nb) * q_blocks;
  if (tiles >= (1u << 24)) return;
  const bool wide = h->d == DVM_ATTN_D;
  // Time of the kernel whose waves divide the queries, in us: one 64-key block behind the other, two workgroups share a
  // compute unit when there are more than compute units, and together they fetch K and V at some 3.6 TB/s (a barrier
  // ends every block).
  const double q_rounds = prog_->grid <= cus ? 1.0 : 1.6 * std::ceil(static_cast<double>(prog_->grid) / static_cast<double>(2 * cus));
  const double t_queries = std::max(3.5 + q_rounds * ((h->skv + DVM_ATTN_BKV - 1) / DVM_ATTN_BKV) * (wide ? 2.0 : 1.3),
                                    static_cast<double>(h->nb) * h->skv * h->d * 4.0 / 3.6e6);
  // Time of a division into `n` parts: rounds of workgroups, per round the steps of its waves (four blocks a step), a step
  // bound by latency and compute (more with a full chip) or by what the workgroups of a round fetch together, 64 KB a step
  // and compute unit at 5.5 TB/s, once for the query tiles of a head (L2); a merge costs its launch, a trip per part and the
  // partial outputs' way through memory.
  auto t_keys = [&](uint32_t n) {
    const double steps = std::ceil(((blocks + n - 1) / n) / static_cast<double>(DVM_ATTN_KEYS_WAVES));
    const uint64_t wgs = tiles * n;
    auto round = [&](double fill) { return std::max(3.2 + steps * (wide ? 1.3 : 0.87) * (1.0 + 0.6 * fill), 1.0 + steps * 3.05 * fill / q_blocks); };
    double us = static_cast<double>(wgs / slots) * round(1.0);
    if (wgs % slots != 0) us += round(static_cast<double>(wgs % slots) / static_cast<double>(slots));
    if (n > 1) us += 6.0 + 0.35 * n + static_cast<double>(h->nb) * n * h->sq * (h->d + 2) * 8.0 / 3.0e6;
    return us;
  };
  // What parts leave in memory stays a small share of the static workspace (DVM_HIP_STATIC_WS_BYTES), beside what the
  // sub-kernels before this one take. (Those behind it are not laid out yet: RunOnce compiles the kernel again without
  // parts when it is they that no longer fit.)
  size_t taken = 0;
  for (size_t bytes : k_->ws_sizes_) taken += (bytes + 255) & ~static_cast<size_t>(255);
  auto part_bytes = [&](uint32_t n) { return static_cast<size_t>(h->nb) * n * h->sq * (h->d + 2) * 4; };
  uint32_t parts = 1;
  if (forced > 1) {
    parts = std::min<uint32_t>(static_cast<uint32_t>(forced), (blocks + DVM_ATTN_KEYS_WAVES - 1) / DVM_ATTN_KEYS_WAVES);
  } else if (forced < 0) {
    double best = t_keys(1);
    const uint32_t most = key_parts_allowed_ ? std::min<uint32_t>(32, (blocks + DVM_ATTN_KEYS_WAVES - 1) / DVM_ATTN_KEYS_WAVES) : 1;
    for (uint32_t n = 2; n <= most; ++n) {
      if (part_bytes(n) > kPartBytes || taken + part_bytes(n) > DVM_HIP_STATIC_WS_BYTES) break;
      const double us = t_keys(n);
      if (us < best) {
        best = us;
        parts = n;
      }
    }
    // Where the estimates are within a fifth and a microsecond the query kernel stays: each key block is read from local memory
    // once for 32 queries of a wave there, and for 32 queries of the workgroup here. Measured on MI355X in us (all launches of
    // a call, by events), waves divide queries / keys (the parts this rule picks): [16,32] heads, 1 query, 1999 keys, D 128:
    // 138 / 95 (1); [1,4], 1, 4096, 128: 104 / 16 (11; undivided 40); [1,32], 8, 4096, 64: 80 / 15 (8; undivided 32); [1,4],
    // 2000, 2000, 128: 65 / 32 (1); [2,8], 500, 1000, 64: 27 / 14 (1); and where the query kernel stays [4,16], 1000, 1000,
    // 128: 49 / 133 (1); [8,32], 100, 200, 128: 17 / 31 (1).
    if (best > 0.8 * t_queries - 1.0) return;
  }
  uint32_t part_blocks = (blocks + parts - 1) / parts;
  part_blocks = std::min<uint32_t>(blocks, (part_blocks + DVM_ATTN_KEYS_WAVES - 1) / DVM_ATTN_KEYS_WAVES * DVM_ATTN_KEYS_WAVES);
  parts = (blocks + part_blocks - 1) / part_blocks;
  h->q_blocks = q_blocks;
  h->kv_parts = parts;
  h->part_blocks = part_blocks;
  prog_->threads = 64 * DVM_ATTN_KEYS_WAVES;
  prog_->lds_bytes = DVM_ATTN_KEYS_LDS_BYTES_D(h->d);
  prog_->grid = static_cast<uint32_t>(tiles * parts);
  if (parts == 1) return;
  Program::Patch pp;
  pp.word = static_cast<uint32_t>(offsetof(VAttnHeader, part_addr) / 8);
  pp.op_id = -1;
  pp.ws_slot = static_cast<int>(k_->ws_sizes_.size());
  pp.role = Program::kPatchPlain;
  k_->ws_sizes_.push_back(part_bytes(parts));
  key_parts_bytes_ += (part_bytes(parts) + 255) & ~static_cast<size_t>(255);
  prog_->patches.push_back(pp);
  const Program first = *prog_;
  k_->programs_.push_back(first);
  prog_ = &k_->programs_.back();
  h = reinterpret_cast<VAttnHeader *>(prog_->blob.w);
  h->merge = 1;
  prog_->lds_bytes = 0;
  prog_->grid = static_cast<uint32_t>((static_cast<uint64_t>(h->nb) * h->sq * (h->d / 4) + prog_->threads - 1) / prog_->threads);
  prog_->fills.clear();
}
}  // namespace dvm
