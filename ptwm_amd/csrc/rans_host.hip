// rans_host.hip -- host orchestration of the rans_ilv encoder.
//
// Per call, any number of planes: histogram kernel and frequency tables
// (ilv_plane_tables, shared with huff_ilv) -> size kernel (word counts per
// block, and the words of the first kRilvKeepBlocks) -> host layout and header
// / offset-table uploads -> the blocks copied to their places, or encoded
// again past kRilvKeepBlocks.  Each plane takes the smallest payload form
// (ilv_choose_form): coded, packed nibbles or stored.  Decode runs through
// ilv_decode_tensors (family kFamilyRans).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "ilv_host.h"
#include "rans_ilv.h"
#include "runtime.h"

namespace ptwm {

// Blocks whose words the size pass keeps: 1032 MiB of scratch at most, for
// 512 MiB of planes.  Blocks past them, and all where the scratch cannot be
// had, are encoded twice.
constexpr uint32_t kRilvKeepBlocks = 32 << 10;

static inline uint64_t align_up(uint64_t v, uint64_t a) { return (v + a - 1) / a * a; }

// A lower bound of the coded payload's bytes, from `bits`, the sum over the
// symbols of 11 - log2 f - 2.25e-5 f.  A lane's state x lies in [2^16, 2^32)
// and a step multiplies it by 2^11 / f, except that rounding x / f down loses
// a factor of at most 1 + f / x: 2.25e-5 f bits at x >= 2^16, and where a word
// left just before, log2(33 / 32) (x >= 32 f) twice, as the shift rounds too.
// So each lane of a block sheds at least (its bits - 16) / 16.0888 words.
static uint64_t rans_ilv_least(uint64_t bits, uint64_t n_blocks, uint32_t head_len) {
  const double words = std::max(0.0, ((double)bits - 1024.0 * (double)n_blocks) / 16.1);
  return align_up(5 + (uint64_t)head_len, 4) + 4 * (n_blocks + 1) + kRilvBlockHead * n_blocks + (uint64_t)(2.0 * words);
}

int64_t rilv_encode_planes(DevCtx& ctx, const uint64_t* src, const uint64_t* n, uint32_t np, uint64_t out_dev,
                           uint64_t out_cap, bool identity_fallback, IlvEncResult* res, uint64_t* needed,
                           const uint8_t* counted) {
  hipStream_t s = ctx.stream;
  if (np == 0) return 0;
  for (uint32_t p = 0; p < np; ++p)
    if ((src[p] & 15u) != 0 || n[p] > 0xFFFFFFFFull) return kInvalidInput;
  std::vector<IlvEncPlane> hp(np);
  uint64_t max_n = 0;
  for (uint32_t p = 0; p < np; ++p) {
    hp[p] = IlvEncPlane{src[p], n[p], p, counted ? counted[p] : 0u};
    max_n = std::max(max_n, n[p]);
  }
  // ---- frequency tables (code_tables.hip): per symbol f | cum << 16 ----
  const TableInfo* info = nullptr;
  if (int64_t rc = ilv_plane_tables(ctx, hp, max_n, kTableRansIlv, counted != nullptr, &info); rc != kOk) return rc;
  std::vector<bool> codable(np, false);
  for (uint32_t p = 0; p < np; ++p) {
    if (n[p] == 0 || !info[p].ok) continue;
    // a plane whose coded payload cannot be shorter than the stored or packed
    // one is not sized: ilv_choose_form would not take it, and the size pass
    // is a whole run of the encoder.  The 11-bit frequencies of a plane of
    // mantissa bytes cost more than 8 bits a symbol, so these planes end
    // here (two bf16 layers, 872 MB: 1763 to 1453 us; MXFP4 14336x2048: 281 to
    // 243 us)
    const uint64_t nb = (n[p] + kIlvBlock - 1) / kIlvBlock;
    const uint64_t stored = n[p] + 1, packed = kPackedHeadBytes + (n[p] + 1) / 2;
    const uint64_t other = info[p].n_sym <= 16 && packed < stored ? packed : stored;
    codable[p] = rans_ilv_least(info[p].bits[0], nb, info[p].head_len) < other;
  }
  // ---- size pass over every block of every codable plane ----
  std::vector<RilvEncBlock> blocks;
  std::vector<uint32_t> first_block(np, 0), nbs(np, 0);
  for (uint32_t p = 0; p < np; ++p) {
    first_block[p] = (uint32_t)blocks.size();
    if (!codable[p]) continue;
    nbs[p] = (uint32_t)((n[p] + kIlvBlock - 1) / kIlvBlock);
    for (uint32_t b = 0; b < nbs[p]; ++b) blocks.push_back(RilvEncBlock{0, p, b, (uint32_t)blocks.size(), 0});
  }
  const uint32_t nblk = (uint32_t)blocks.size();
  PTWM_HIP_TRY(ctx.h_sizes.ensure(nblk * sizeof(uint32_t)));
  uint32_t* const bwords = static_cast<uint32_t*>(ctx.h_sizes.ptr);
  uint32_t kept = std::min(nblk, kRilvKeepBlocks);
  if (nblk) {
    // all that the encode cannot do without, the last pass's upload at its
    // largest included, before the blocks' words (DeviceBuffer::spare)
    PTWM_HIP_TRY(ctx.enc_blocks.ensure(nblk * sizeof(RilvEncBlock)));
    PTWM_HIP_TRY(ctx.enc_block_bytes.ensure(nblk * sizeof(uint32_t)));
    size_t pack = ilv_upload_bound(np, nblk * sizeof(RilvEncBlock));
    for (uint32_t p = 0; p < np; ++p)
      if (codable[p]) pack += align_up(5 + (uint64_t)info[p].head_len, 4) + 4 * ((uint64_t)nbs[p] + 1);
    PTWM_HIP_TRY(ctx.enc_pack.ensure(pack));
    if (kept && ctx.enc_keep.ensure(kept * kRilvKeepBytes) != hipSuccess) {
      (void)hipGetLastError();
      kept = 0;
    }
    PTWM_HIP_TRY(ctx.h_enc.ensure(nblk * sizeof(RilvEncBlock)));
    std::memcpy(ctx.h_enc.ptr, blocks.data(), nblk * sizeof(RilvEncBlock));
    PTWM_HIP_TRY(
        hipMemcpyAsync(ctx.enc_blocks.ptr, ctx.h_enc.ptr, nblk * sizeof(RilvEncBlock), hipMemcpyHostToDevice, s));
    PTWM_HIP_TRY(launch_rilv_size(static_cast<const IlvEncPlane*>(ctx.enc_planes.ptr),
                                  static_cast<const RilvEncBlock*>(ctx.enc_blocks.ptr), nblk, kept,
                                  static_cast<const uint32_t*>(ctx.enc_codes.ptr),
                                  static_cast<uint32_t*>(ctx.enc_block_bytes.ptr),
                                  static_cast<uint8_t*>(ctx.enc_keep.ptr), s));
    PTWM_HIP_TRY(hipMemcpyAsync(bwords, ctx.enc_block_bytes.ptr, nblk * 4, hipMemcpyDeviceToHost, s));
    PTWM_HIP_TRY(hipStreamSynchronize(s));
  }
  // ---- layout: payloads at 256-byte aligned offsets ----
  uint64_t off = 0;
  std::vector<uint64_t> head(np, 0);
  std::vector<uint32_t> form(np, kFormStored);
  for (uint32_t p = 0; p < np; ++p) {
    off = align_up(off, 256);
    res[p].offset = off;
    uint64_t pay = 0;
    bool codable_p = codable[p];
    if (codable_p) {
      uint64_t d = 0;
      for (uint32_t b = 0; b < nbs[p]; ++b) d += align_up(kRilvBlockHead + 2ull * bwords[first_block[p] + b], 4);
      head[p] = align_up(5 + (uint64_t)info[p].head_len, 4);
      pay = head[p] + 4ull * (nbs[p] + 1) + d;
      codable_p = d <= 0xFFFFFFFFull;
    }
    form[p] = ilv_choose_form(n[p], info[p].n_sym <= 16, codable_p, pay, identity_fallback, &res[p].len);
    res[p].coded = form[p] == kFormCoded ? 1 : 0;
    res[p].codec = form[p] == kFormIdentity ? kCodecIdentity : kCodecRansIlv;
    off += res[p].len;
  }
  const uint64_t total = off;
  if (total > out_cap) {
    if (needed) *needed = total;
    return kBufferTooSmall;
  }
  // ---- headers, offset tables, stored / packed planes, block destinations:
  // one upload ----
  size_t live = 0, n_kept = 0;  // blocks of coded planes, and those whose words are there
  std::vector<uint64_t> head_len(np, 0);
  for (uint32_t p = 0; p < np; ++p)
    if (res[p].coded) {
      head_len[p] = head[p] + 4ull * (nbs[p] + 1);
      live += nbs[p];
    }
  IlvUpload u;
  if (int64_t rc = ilv_upload_begin(ctx, src, n, np, out_dev, res, form.data(), head_len.data(),
                                    live * sizeof(RilvEncBlock), u);
      rc != kOk)
    return rc;
  RilvEncBlock* hblk = reinterpret_cast<RilvEncBlock*>(u.host + u.blocks);
  for (uint32_t p = 0; p < np; ++p) {
    if (!res[p].coded) continue;
    uint8_t* const h = u.host + u.head[p];
    h[0] = 1;
    const uint32_t nn = (uint32_t)n[p];
    std::memcpy(h + 1, &nn, 4);
    std::memcpy(h + 5, info[p].head, info[p].head_len);
    uint32_t* tab = reinterpret_cast<uint32_t*>(h + head[p]);
    uint64_t acc = 0;
    const uint64_t data_dev = out_dev + res[p].offset + head_len[p];
    for (uint32_t b = 0; b < nbs[p]; ++b) {
      const uint32_t i = first_block[p] + b;
      tab[b] = (uint32_t)acc;
      *hblk++ = RilvEncBlock{data_dev + acc, p, b, i, 0};
      n_kept += i < kept;  // (i rises along the list)
      acc += align_up(kRilvBlockHead + 2ull * bwords[i], 4);
    }
    tab[nbs[p]] = (uint32_t)acc;
  }
  if (int64_t rc = ilv_upload_send(ctx, u); rc != kOk) return rc;
  if (live) {
    const RilvEncBlock* const bd = reinterpret_cast<const RilvEncBlock*>(u.dev + u.blocks);
    const uint32_t* const words = static_cast<const uint32_t*>(ctx.enc_block_bytes.ptr);
    PTWM_HIP_TRY(
        launch_rilv_place(bd, (uint32_t)n_kept, words, static_cast<const uint8_t*>(ctx.enc_keep.ptr), s));
    PTWM_HIP_TRY(launch_rilv_encode(static_cast<const IlvEncPlane*>(ctx.enc_planes.ptr), bd + n_kept,
                                    (uint32_t)(live - n_kept), static_cast<const uint32_t*>(ctx.enc_codes.ptr), words,
                                    s));
  }
  PTWM_HIP_TRY(hipStreamSynchronize(s));
  return (int64_t)total;
}

}  // namespace ptwm
