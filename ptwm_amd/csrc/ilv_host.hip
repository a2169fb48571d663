// ilv_host.hip -- host orchestration of the huff_ilv encoder and decoder.
//
// Encode (per call, any number of planes): histogram kernel -> code tables
// (code_tables.hip) -> size kernel -> host prefix sums and payload
// layout -> encode kernel plus header / offset-table uploads.  Each plane
// takes the smallest payload form (ilv_choose_form): coded, packed nibbles
// or stored.
//
// Decode: tensors are grouped by chain and decoded with one fused launch per
// chain (ilv_decode_kernel<chain>): persistent workgroups (as many as fit on
// the device at the launch's LDS size) over 4-block tiles.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "huff_ilv.h"
#include "ilv_host.h"
#include "integrity.h"
#include "rans_ilv.h"
#include "runtime.h"

namespace ptwm {

static inline uint64_t align_up(uint64_t v, uint64_t a) { return (v + a - 1) / a * a; }

uint32_t ilv_choose_form(uint64_t n, bool nibbles, bool codable, uint64_t coded_len, bool identity_fallback,
                         uint64_t* len) {
  const uint64_t stored = n + 1, packed = kPackedHeadBytes + (n + 1) / 2;
  const bool pack_ok = nibbles && packed < stored;
  const uint64_t other = pack_ok ? packed : stored;
  uint32_t form = kFormStored;
  uint64_t l = stored;
  if (codable && coded_len < other) {
    form = kFormCoded;
    l = coded_len;
  } else if (pack_ok) {
    form = kFormPacked;
    l = packed;
  }
  if (identity_fallback && (form == kFormStored || l >= n)) {
    form = kFormIdentity;
    l = n;
  }
  *len = l;
  return form;
}

int64_t ilv_upload_begin(DevCtx& ctx, const uint64_t* src, const uint64_t* n, uint32_t np, uint64_t out_dev,
                         const IlvEncResult* res, const uint32_t* form, const uint64_t* head_len, size_t block_bytes,
                         IlvUpload& u) {
  u = IlvUpload{};
  std::vector<IlvPackJob> pack;
  std::vector<IlvStoreJob> store, heads;  // heads: src filled in below
  std::vector<uint32_t> head_of;
  for (uint32_t p = 0; p < np; ++p) {
    const uint64_t dst = out_dev + res[p].offset;
    if (form[p] == kFormIdentity || form[p] == kFormStored) {
      const uint32_t shift = form[p] == kFormStored ? 1u : 0u;
      if (n[p] + shift == 0) continue;
      store.push_back(IlvStoreJob{src[p], dst, n[p], shift, 0});
      u.max_store = std::max(u.max_store, n[p] + shift);
      continue;
    }
    if (form[p] == kFormPacked) {
      pack.push_back(IlvPackJob{src[p], dst + kPackedHeadBytes, n[p]});
      u.max_pack = std::max(u.max_pack, n[p]);
    }
    const uint64_t len = form[p] == kFormPacked ? kPackedHeadBytes : head_len[p];
    heads.push_back(IlvStoreJob{0, dst, len, 0, 0});
    head_of.push_back(p);
    u.max_head = std::max(u.max_head, len);
  }
  size_t at = 0;
  auto place = [&at](size_t bytes) {
    const size_t a = at;
    at = align_up(at + bytes, 16);
    return a;
  };
  u.pack_jobs = place(pack.size() * sizeof(IlvPackJob));
  u.store_jobs = place(store.size() * sizeof(IlvStoreJob));
  u.head_jobs = place(heads.size() * sizeof(IlvStoreJob));
  const size_t first_head = at;
  u.head.assign(np, 0);
  for (size_t i = 0; i < heads.size(); ++i) u.head[head_of[i]] = place(heads[i].n);
  u.blocks = place(block_bytes);
  u.bytes = at;
  u.n_pack = (uint32_t)pack.size();
  u.n_store = (uint32_t)store.size();
  u.n_head = (uint32_t)heads.size();
  if (!u.bytes) return kOk;
  PTWM_HIP_TRY(ctx.enc_pack.ensure(u.bytes));
  PTWM_HIP_TRY(ctx.h_enc.ensure(u.bytes));
  u.host = static_cast<uint8_t*>(ctx.h_enc.ptr);
  u.dev = static_cast<uint8_t*>(ctx.enc_pack.ptr);
  for (size_t i = 0; i < heads.size(); ++i)
    heads[i].src = reinterpret_cast<uint64_t>(u.dev) + u.head[head_of[i]];
  std::copy(pack.begin(), pack.end(), reinterpret_cast<IlvPackJob*>(u.host + u.pack_jobs));
  std::copy(store.begin(), store.end(), reinterpret_cast<IlvStoreJob*>(u.host + u.store_jobs));
  std::copy(heads.begin(), heads.end(), reinterpret_cast<IlvStoreJob*>(u.host + u.head_jobs));
  std::memset(u.host + first_head, 0, u.blocks - first_head);
  for (const uint32_t p : head_of)
    if (form[p] == kFormPacked) {
      uint8_t* const h = u.host + u.head[p];
      h[0] = 2;
      const uint32_t nn = (uint32_t)n[p];
      std::memcpy(h + 1, &nn, 4);
    }
  return kOk;
}

size_t ilv_upload_bound(uint32_t np, size_t block_bytes) {
  // per plane a pack and a head job or a store job, and a head; each piece
  // rounded up to 16
  return np * (sizeof(IlvPackJob) + 2 * sizeof(IlvStoreJob) + align_up(kPackedHeadBytes, 16) + 16) + 4 * 16 +
         align_up(block_bytes, 16);
}

int64_t ilv_upload_send(DevCtx& ctx, const IlvUpload& u) {
  if (!u.bytes) return kOk;
  hipStream_t s = ctx.stream;
  PTWM_HIP_TRY(hipMemcpyAsync(u.dev, u.host, u.bytes, hipMemcpyHostToDevice, s));
  PTWM_HIP_TRY(launch_ilv_store(reinterpret_cast<const IlvStoreJob*>(u.dev + u.head_jobs), u.n_head, u.max_head, s));
  PTWM_HIP_TRY(launch_ilv_pack(reinterpret_cast<const IlvPackJob*>(u.dev + u.pack_jobs), u.n_pack, u.max_pack, s));
  PTWM_HIP_TRY(launch_ilv_store(reinterpret_cast<const IlvStoreJob*>(u.dev + u.store_jobs), u.n_store, u.max_store, s));
  return kOk;
}

uint32_t* ilv_hist_begin(DevCtx& ctx, uint32_t np) {
  const size_t bytes = (size_t)np * 256 * sizeof(uint32_t);
  if (ctx.enc_hist.ensure(bytes) != hipSuccess || hipMemsetAsync(ctx.enc_hist.ptr, 0, bytes, ctx.stream) != hipSuccess)
    return nullptr;
  return static_cast<uint32_t*>(ctx.enc_hist.ptr);
}

int64_t ilv_plane_tables(DevCtx& ctx, const std::vector<IlvEncPlane>& planes, uint64_t max_n, uint32_t kind,
                         bool begun, const TableInfo** info) {
  hipStream_t s = ctx.stream;
  const uint32_t np = (uint32_t)planes.size();
  const size_t b_pl = np * sizeof(IlvEncPlane), b_tj = np * sizeof(TableJob);
  PTWM_HIP_TRY(ctx.enc_planes.ensure(b_pl + b_tj));
  if (!begun && !ilv_hist_begin(ctx, np)) return kInternal;
  PTWM_HIP_TRY(ctx.enc_codes.ensure(np * 256 * sizeof(uint32_t)));
  PTWM_HIP_TRY(ctx.h_enc.ensure(b_pl + b_tj));
  PTWM_HIP_TRY(ctx.h_tables.ensure(np * sizeof(TableInfo)));
  uint8_t* const h = static_cast<uint8_t*>(ctx.h_enc.ptr);
  std::memcpy(h, planes.data(), b_pl);
  TableJob* const tj = reinterpret_cast<TableJob*>(h + b_pl);
  for (uint32_t p = 0; p < np; ++p) tj[p] = TableJob{kind, p, 1, 0};
  uint8_t* const d = static_cast<uint8_t*>(ctx.enc_planes.ptr);
  uint32_t* const hist = static_cast<uint32_t*>(ctx.enc_hist.ptr);
  TableInfo* const out = static_cast<TableInfo*>(ctx.h_tables.ptr);
  PTWM_HIP_TRY(hipMemcpyAsync(d, h, b_pl + b_tj, hipMemcpyHostToDevice, s));
  if (!std::all_of(planes.begin(), planes.end(), [](const IlvEncPlane& p) { return p.counted != 0; }))
    PTWM_HIP_TRY(launch_ilv_hist(reinterpret_cast<const IlvEncPlane*>(d), np, max_n, hist, s));
  PTWM_HIP_TRY(launch_code_tables(reinterpret_cast<const TableJob*>(d + b_pl), np, hist,
                                  static_cast<uint32_t*>(ctx.enc_codes.ptr), nullptr, out, s));
  PTWM_HIP_TRY(hipStreamSynchronize(s));
  *info = out;
  return kOk;
}

int64_t ilv_encode_planes(DevCtx& ctx, const uint64_t* src, const uint64_t* n, uint32_t np, uint64_t out_dev,
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
  // ---- code tables (code_tables.hip) ----
  const TableInfo* info = nullptr;
  if (int64_t rc = ilv_plane_tables(ctx, hp, max_n, kTableIlv, counted != nullptr, &info); rc != kOk) return rc;
  std::vector<uint8_t> codable(np, 0);
  for (uint32_t p = 0; p < np; ++p) {
    if (n[p] == 0 || !info[p].ok) continue;
    // a coded payload is at least its header, offset table, lane counts
    // and ceil(code bits / 8): a plane for which that is not shorter than
    // the stored or packed form is not sized (the form choice below would
    // not take the coded form)
    const uint64_t nb = (n[p] + kIlvBlock - 1) / kIlvBlock;
    const uint64_t lower = align_up(5 + (uint64_t)info[p].head_len, 4) + 4 * (nb + 1) + 64 * nb + (info[p].bits[0] + 7) / 8;
    const uint64_t stored = n[p] + 1, packed = kPackedHeadBytes + (n[p] + 1) / 2;
    const uint64_t other = info[p].n_sym <= 16 && packed < stored ? packed : stored;
    codable[p] = lower < other;
  }
  // ---- size pass over every block of every codable plane ----
  std::vector<IlvEncBlock> blocks;
  std::vector<uint32_t> first_block(np, 0), nbs(np, 0);
  for (uint32_t p = 0; p < np; ++p) {
    first_block[p] = (uint32_t)blocks.size();
    if (!codable[p]) continue;
    nbs[p] = (uint32_t)((n[p] + kIlvBlock - 1) / kIlvBlock);
    for (uint32_t b = 0; b < nbs[p]; ++b) blocks.push_back(IlvEncBlock{0, p, b, 0, 0});
  }
  const uint32_t nblk = (uint32_t)blocks.size();
  PTWM_HIP_TRY(ctx.h_sizes.ensure(nblk * sizeof(uint32_t)));
  uint32_t* const bbytes = static_cast<uint32_t*>(ctx.h_sizes.ptr);
  if (nblk) {
    PTWM_HIP_TRY(ctx.enc_blocks.ensure(nblk * sizeof(IlvEncBlock)));
    PTWM_HIP_TRY(ctx.enc_lane_words.ensure((size_t)nblk * 64));
    PTWM_HIP_TRY(ctx.enc_block_bytes.ensure(nblk * sizeof(uint32_t)));
    PTWM_HIP_TRY(ctx.h_enc.ensure(nblk * sizeof(IlvEncBlock)));
    std::memcpy(ctx.h_enc.ptr, blocks.data(), nblk * sizeof(IlvEncBlock));
    PTWM_HIP_TRY(hipMemcpyAsync(ctx.enc_blocks.ptr, ctx.h_enc.ptr, nblk * sizeof(IlvEncBlock), hipMemcpyHostToDevice,
                                s));
    PTWM_HIP_TRY(launch_ilv_size(static_cast<const IlvEncPlane*>(ctx.enc_planes.ptr),
                                 static_cast<const IlvEncBlock*>(ctx.enc_blocks.ptr), nblk,
                                 static_cast<const uint32_t*>(ctx.enc_codes.ptr),
                                 static_cast<uint8_t*>(ctx.enc_lane_words.ptr),
                                 static_cast<uint32_t*>(ctx.enc_block_bytes.ptr), s));
    PTWM_HIP_TRY(hipMemcpyAsync(bbytes, ctx.enc_block_bytes.ptr, nblk * 4, hipMemcpyDeviceToHost, s));
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
      for (uint32_t b = 0; b < nbs[p]; ++b) d += bbytes[first_block[p] + b];
      head[p] = align_up(5 + (uint64_t)info[p].head_len, 4);
      pay = head[p] + 4ull * (nbs[p] + 1) + d;
      codable_p = d <= 0xFFFFFFFFull;
    }
    form[p] = ilv_choose_form(n[p], info[p].n_sym <= 16, codable_p, pay, identity_fallback, &res[p].len);
    res[p].coded = form[p] == kFormCoded ? 1 : 0;
    res[p].codec = form[p] == kFormIdentity ? kCodecIdentity : kCodecHuffIlv;
    off += res[p].len;
  }
  const uint64_t total = off;
  if (total > out_cap) {
    if (needed) *needed = total;
    return kBufferTooSmall;
  }
  // ---- headers, offset tables and block destinations: one upload ----
  // (only blocks of coded planes are written; lw keeps the size-pass index)
  size_t live = 0;
  std::vector<uint64_t> head_len(np, 0);
  for (uint32_t p = 0; p < np; ++p)
    if (res[p].coded) {
      head_len[p] = head[p] + 4ull * (nbs[p] + 1);
      live += nbs[p];
    }
  IlvUpload u;
  if (int64_t rc = ilv_upload_begin(ctx, src, n, np, out_dev, res, form.data(), head_len.data(),
                                    live * sizeof(IlvEncBlock), u);
      rc != kOk)
    return rc;
  IlvEncBlock* hblk = reinterpret_cast<IlvEncBlock*>(u.host + u.blocks);
  uint32_t max_words = 0;
  for (uint32_t p = 0; p < np; ++p) {
    if (!res[p].coded) continue;
    uint8_t* h = u.host + u.head[p];
    h[0] = 1;
    uint32_t nn = (uint32_t)n[p];
    std::memcpy(h + 1, &nn, 4);
    std::memcpy(h + 5, info[p].head, info[p].head_len);
    uint32_t* tab = reinterpret_cast<uint32_t*>(h + head[p]);
    uint64_t acc = 0;
    const uint64_t data_dev = out_dev + res[p].offset + head_len[p];
    for (uint32_t b = 0; b < nbs[p]; ++b) {
      const uint32_t i = first_block[p] + b;
      tab[b] = (uint32_t)acc;
      *hblk++ = IlvEncBlock{data_dev + acc, p, b, i, 0};
      acc += bbytes[i];
      max_words = std::max(max_words, bbytes[i] >= 64 ? (bbytes[i] - 64) / 4 : 0u);
    }
    tab[nbs[p]] = (uint32_t)acc;
  }
  if (int64_t rc = ilv_upload_send(ctx, u); rc != kOk) return rc;
  // LDS for the largest block's words, within the cap (larger blocks are
  // written lane by lane)
  const uint32_t stage_words = std::min<uint32_t>(kIlvEncStageMax, (max_words + 3) & ~3u);
  PTWM_HIP_TRY(launch_ilv_encode(static_cast<const IlvEncPlane*>(ctx.enc_planes.ptr),
                                 reinterpret_cast<const IlvEncBlock*>(u.dev + u.blocks), (uint32_t)live,
                                 static_cast<const uint32_t*>(ctx.enc_codes.ptr),
                                 static_cast<const uint8_t*>(ctx.enc_lane_words.ptr), stage_words, s));
  PTWM_HIP_TRY(hipStreamSynchronize(s));
  return (int64_t)total;
}

int64_t ilv_decode_tensors(DevCtx& ctx, const std::vector<IlvTensor>& tensors_in, uint32_t n_acc,
                           std::vector<uint32_t>& crc, std::vector<uint32_t>& flagged, bool all_slots) {
  hipStream_t s = ctx.stream;
  if (tensors_in.empty()) return kOk;
  std::vector<IlvTensor> tensors = tensors_in;
  const size_t nt = tensors.size();
  if (ctx.cu_count <= 0) {
    PTWM_HIP_TRY(hipDeviceGetAttribute(&ctx.cu_count, hipDeviceAttributeMultiprocessorCount, ctx.dev));
    if (ctx.cu_count <= 0) ctx.cu_count = 1;
  }
  // Coded payloads are read as 32-bit words: copy the ones that do not
  // start on a 4-byte boundary to aligned scratch first.
  uint64_t realign_bytes = 0;
  for (const IlvTensor& T : tensors)
    for (uint32_t p = 0; p < T.n_planes; ++p)
      if (T.planes[p].coded && (T.planes[p].base & 3u)) realign_bytes = align_up(realign_bytes + T.planes[p].len, 256);
  if (realign_bytes) {
    // one batched copy for all of them (chunk frames put most payloads of a
    // chunked plane off 4-byte boundaries)
    PTWM_HIP_TRY(ctx.ilv_realign.ensure(realign_bytes));
    std::vector<IlvStoreJob> jobs;
    uint64_t off = 0, max_n = 0;
    for (IlvTensor& T : tensors)
      for (uint32_t p = 0; p < T.n_planes; ++p) {
        IlvPlane& P = T.planes[p];
        if (!P.coded || !(P.base & 3u)) continue;
        const uint64_t dst = reinterpret_cast<uint64_t>(ctx.ilv_realign.ptr) + off;
        jobs.push_back(IlvStoreJob{P.base, dst, P.len, 0, 0});
        max_n = P.len > max_n ? P.len : max_n;
        P.base = dst;
        off = align_up(off + P.len, 256);
      }
    const size_t jb = jobs.size() * sizeof(IlvStoreJob);
    PTWM_HIP_TRY(ctx.realign_jobs.ensure(jb));
    PTWM_HIP_TRY(ctx.h_realign.ensure(jb));
    std::memcpy(ctx.h_realign.ptr, jobs.data(), jb);
    PTWM_HIP_TRY(hipMemcpyAsync(ctx.realign_jobs.ptr, ctx.h_realign.ptr, jb, hipMemcpyHostToDevice, s));
    PTWM_HIP_TRY(launch_ilv_realign(static_cast<const IlvStoreJob*>(ctx.realign_jobs.ptr), (uint32_t)jobs.size(),
                                    max_n, s));
  }
  // One persistent launch per chain present.  Per launch: the tensor list,
  // its 4-block tile prefix sums, the LDS table slots (most coded planes of
  // any tensor) and the room for blocks' streams: estimated block sizes
  // (coded payload words per block, +2%, rounded up), capped by the workgroup
  // LDS budget.  rans_ilv: staging words per wavefront, the largest of any
  // tensor; huff_ilv: the pool's bytes, the most that any tensor's tables and
  // staging take together.  Blocks above it take the kernel's global-memory
  // path.
  struct Launch {
    uint32_t family, chain, first, m, slots, room, grid;
    bool crc;  // some tensor of the launch has plane CRCs
  };
  std::vector<Launch> launches;
  // The launch chain codes of a family: one per chain present, except that
  // huff_ilv nibble-split and passthrough tensors (MXFP4 weights and their
  // scales) share one two-chain launch.
  bool pair_ok = false;
  {
    bool has5 = false, has6 = false;
    for (const IlvTensor& T : tensors) {
      if (T.family != kFamilyHuff || T.n == 0) continue;
      has5 |= T.chain == kChainNibbleSplit;
      has6 |= T.chain == kChainPassthrough;
    }
    pair_ok = has5 && has6;
  }
  auto launch_codes = [&](uint32_t fam) {
    std::vector<uint32_t> codes{kChainIeee16Split2, kChainIeee32Split4, kChainE4m3Nibble, kChainE5m2Nibble};
    if (fam == kFamilyHuff && pair_ok) {
      codes.push_back(kIlvPairNibblePass);
    } else {
      codes.push_back(kChainNibbleSplit);
      codes.push_back(kChainPassthrough);
    }
    return codes;
  };
  std::vector<uint32_t> idx;  // per launch: [m + 1 prefix][m tensor indexes]
  // Within a launch, the tensors whose tiles build decode tables come first:
  // the workgroups of the last tiles start a few microseconds late and set
  // up under the others' streaming traffic, so the tiles with the longest
  // setup (table builds and staging) go to the first workgroups (MXFP4: the
  // coded E8M0 scales ahead of the packed weights).
  std::vector<uint32_t> order;
  order.reserve(nt);
  for (int pass = 0; pass < 2; ++pass)
    for (uint32_t ti = 0; ti < nt; ++ti) {
      const IlvTensor& T = tensors[ti];
      bool tables = false;
      for (uint32_t p = 0; p < T.n_planes; ++p) {
        const IlvPlane& P = T.planes[p];
        tables |= P.coded && P.len != T.n + 1 && P.len != kPackedHeadBytes + (T.n + 1) / 2;
      }
      if (tables == (pass == 0)) order.push_back(ti);
    }
  // Tensors without plane CRCs go along in a launch with them, whose kernel
  // takes the CRCs and drops these; many blocks of them have a launch of their
  // own, which the device starts some 25 us later (512 MiB of bf16 planes
  // beside one tensor with CRCs: huff_ilv 284 to 252 us, rans_ilv 434 to 334).
  constexpr uint64_t kPlainBlocks = 8192;
  uint64_t chain_blocks[2][8][2] = {};  // by family, chain and whether without CRCs
  for (const IlvTensor& T : tensors)
    if (T.family <= kFamilyRans && T.chain < 8)
      chain_blocks[T.family][T.chain][T.crc_ix == kIlvNoCrc] += (T.n + kIlvBlock - 1) / kIlvBlock;
  for (uint32_t fam = kFamilyHuff; fam <= kFamilyRans; ++fam)
  for (uint32_t chain : launch_codes(fam))
  for (const bool plain : {false, true}) {
    uint64_t blocks[2] = {};
    for (uint32_t c = 0; c < 8; ++c)
      if (ilv_code_has(chain, c))
        for (uint32_t k = 0; k < 2; ++k) blocks[k] += chain_blocks[fam][c][k];
    const bool apart = blocks[0] && blocks[1] >= kPlainBlocks;
    if (plain ? !apart : !(blocks[0] + blocks[1])) continue;
    std::vector<uint32_t> tix, tpre{0};
    uint32_t slots = 0;
    uint64_t est = 0, pool = 0, pool_skew = 0;
    bool with_crc = false;
    for (const uint32_t ti : order) {
      const IlvTensor& T = tensors[ti];
      if (T.family != fam || !ilv_code_has(chain, T.chain) || T.n == 0) continue;
      if (apart && (T.crc_ix == kIlvNoCrc) != plain) continue;
      with_crc |= T.crc_ix != kIlvNoCrc;
      const uint64_t nb = (T.n + kIlvBlock - 1) / kIlvBlock;
      // LDS table slots and staging for the planes that may be coded: a
      // native payload of the stored (n + 1) or packed (8 + ceil(n / 2))
      // length is taken as such.  A coded plane of either length finds no
      // slot, and its tensor is decoded again with a slot for every plane
      // (kIlvRetrySlots); its blocks may take the kernel's global-memory path.
      uint32_t need_slots = 0;
      // (skew: huff_ilv nibble chains may carry fixed-length codes, whose
      // equal-length lane streams the kernel skews by up to two words a lane)
      uint64_t words = fam == kFamilyHuff ? 4 : 0, skew = 0;
      for (uint32_t p = 0; p < T.n_planes; ++p) {
        const IlvPlane& P = T.planes[p];
        if (!P.coded) continue;
        if (!all_slots && (P.len == T.n + 1 || P.len == kPackedHeadBytes + (T.n + 1) / 2)) continue;
        ++need_slots;
        const uint64_t per_block = (T.planes[p].len + 4 * nb - 1) / (4 * nb);
        words += align_up(per_block + per_block / 50 + 4, 4);
        skew += fam == kFamilyRans || T.chain == kChainIeee16Split2 || T.chain == kChainIeee32Split4 ? 0 : 128;
      }
      slots = std::max(slots, need_slots);
      est = std::max(est, words);
      if (fam == kFamilyHuff) {
        const uint64_t tables = (uint64_t)need_slots * ilv_slot_bytes(chain);
        pool = std::max(pool, tables + 16 * words);
        pool_skew = std::max(pool_skew, tables + 16 * (words + skew));
      }
      tix.push_back(ti);
      tpre.push_back(tpre.back() + (uint32_t)((nb + kIlvBlocksPerTile - 1) / kIlvBlocksPerTile));
    }
    if (tix.empty()) continue;
    // workgroups per CU with `room` (Launch::room) for the blocks
    const auto occupancy = [&](uint64_t room, int& per_cu) -> int64_t {
      const uint64_t key =
          (uint64_t)chain | ((uint64_t)slots << 12) | (room << 20) | ((uint64_t)with_crc << 61) | ((uint64_t)fam << 62);
      auto it = ctx.ilv_occupancy.find(key);
      if (it != ctx.ilv_occupancy.end()) {
        per_cu = it->second;
        return kOk;
      }
      if (fam == kFamilyHuff) PTWM_HIP_TRY(ilv_decode_occupancy(chain, (uint32_t)room, with_crc, &per_cu));
      else PTWM_HIP_TRY(rilv_decode_occupancy(chain, slots, (uint32_t)room, with_crc, &per_cu));
      ctx.ilv_occupancy[key] = per_cu;
      return kOk;
    };
    int per_cu = 0;
    uint64_t room = 0;
    // The LDS budgets hold without what plane CRCs take on top (blocks that
    // are not staged decode from global memory, several times slower).  The
    // room also holds the payload heads at a tensor's start.
    if (fam == kFamilyHuff) {
      const uint64_t least = (uint64_t)slots * ilv_slot_bytes(chain) + 16 * kIlvHeadWords;
      const uint64_t most = (kIlvMaxLds - ilv_decode_lds_bytes(chain, 0, false)) / kIlvPoolAlign * kIlvPoolAlign;
      if (least > most) return kInternal;
      room = std::min(align_up(std::max(pool, least), kIlvPoolAlign), most);
      if (int64_t rc = occupancy(room, per_cu); rc != kOk) return rc;
      // room for the skew where it does not cost a workgroup per CU
      const uint64_t with_skew = std::min(align_up(std::max(pool_skew, least), kIlvPoolAlign), most);
      int n = 0;
      if (with_skew != room)
        if (int64_t rc = occupancy(with_skew, n); rc != kOk) return rc;
      if (n >= per_cu) room = with_skew;
    } else {
      const uint64_t fixed = rilv_decode_lds_bytes(chain, slots, 0, false);
      const uint64_t cap_words = ((kRilvMaxLds - std::min<uint64_t>(fixed, kRilvMaxLds)) / 16) & ~3ull;
      room = std::min(align_up(std::max<uint64_t>({est, 8, kRilvHeadWords}), 4), cap_words);
      if (room < kRilvHeadWords) return kInternal;
      if (int64_t rc = occupancy(room, per_cu); rc != kOk) return rc;
    }
    if (per_cu < 1) per_cu = 1;
    const uint64_t n_tiles = tpre.back();
    const uint32_t grid = (uint32_t)std::min<uint64_t>(n_tiles, (uint64_t)per_cu * ctx.cu_count);
    launches.push_back(Launch{fam, chain, (uint32_t)idx.size(), (uint32_t)tix.size(), slots, (uint32_t)room, grid, with_crc});
    idx.insert(idx.end(), tpre.begin(), tpre.end());
    idx.insert(idx.end(), tix.begin(), tix.end());
  }
  // Launches of at most kIlvInlineTensors huff_ilv tensors take their
  // descriptors in the kernel arguments; the others read them from one
  // upload: [tensor descriptors][launch index arrays].  The status words are
  // host-coherent: zeroed here, ORed by the kernels, read after the stream
  // has drained (no copy back).
  PTWM_HIP_TRY(ctx.h_ilv_status.ensure(nt * sizeof(uint32_t)));
  uint32_t* const hs = static_cast<uint32_t*>(ctx.h_ilv_status.ptr);
  std::memset(hs, 0, nt * sizeof(uint32_t));
  auto inline_ok = [](const Launch& L) { return L.family == kFamilyHuff && L.m <= kIlvInlineTensors; };
  bool upload = false;
  for (const Launch& L : launches) upload |= !inline_ok(L);
  const size_t off_idx = align_up(nt * sizeof(IlvTensor), 16);
  const size_t args_bytes = off_idx + idx.size() * sizeof(uint32_t);
  uint8_t* d = nullptr;
  if (upload) {
    PTWM_HIP_TRY(ctx.ilv_args.ensure(args_bytes));
    PTWM_HIP_TRY(ctx.h_ilv.ensure(args_bytes));
    uint8_t* h = static_cast<uint8_t*>(ctx.h_ilv.ptr);
    std::memcpy(h, tensors.data(), nt * sizeof(IlvTensor));
    std::memcpy(h + off_idx, idx.data(), idx.size() * sizeof(uint32_t));
    d = static_cast<uint8_t*>(ctx.ilv_args.ptr);
    PTWM_HIP_TRY(hipMemcpyAsync(d, h, args_bytes, hipMemcpyHostToDevice, s));
  }
  if (ctx.profile) {
    PTWM_HIP_TRY(ctx.ensure_events());
    PTWM_HIP_TRY(hipEventRecord(ctx.ev[3], s));
  }
  // the call's last launch with plane CRCs hands their sums over
  CrcArgs crc_args{};
  size_t last_crc = launches.size();
  for (size_t i = 0; i < launches.size(); ++i)
    if (launches[i].crc) last_crc = i;
  if (last_crc < launches.size())
    if (int64_t rc = crc_begin(ctx, n_acc, crc_args); rc != kOk) return rc;
  for (size_t li = 0; li < launches.size(); ++li) {
    const Launch& L = launches[li];
    CrcArgs ca = crc_args;
    if (li != last_crc) ca.n = 0;
    const CrcArgs* const cp = L.crc ? &ca : nullptr;
    const uint32_t* hidx = idx.data() + L.first;  // [m + 1 prefix][m tensor indexes]
    if (inline_ok(L)) {
      IlvInline inl{};
      inl.m = L.m;
      for (uint32_t j = 0; j <= L.m; ++j) inl.tpre[j] = hidx[j];
      for (uint32_t j = 0; j < L.m; ++j) {
        inl.tix[j] = hidx[L.m + 1 + j];
        inl.t[j] = tensors[inl.tix[j]];
      }
      PTWM_HIP_TRY(launch_ilv_decode(L.chain, nullptr, nullptr, nullptr, 0, inl, L.grid, hs, L.slots,
                                     L.room, cp, s));
      continue;
    }
    const uint32_t* base = reinterpret_cast<const uint32_t*>(d + off_idx) + L.first;
    const IlvTensor* td = reinterpret_cast<const IlvTensor*>(d);
    if (L.family == kFamilyHuff)
      PTWM_HIP_TRY(launch_ilv_decode(L.chain, td, base + L.m + 1, base, L.m, IlvInline{}, L.grid, hs, L.slots,
                                     L.room, cp, s));
    else
      PTWM_HIP_TRY(launch_rilv_decode(L.chain, td, base + L.m + 1, base, L.m, L.grid, hs, L.slots,
                                      L.room, cp, s));
  }
  if (ctx.profile) PTWM_HIP_TRY(hipEventRecord(ctx.ev[2], s));
  PTWM_HIP_TRY(hipStreamSynchronize(s));
  if (ctx.profile) {
    float ms = 0;
    PTWM_HIP_TRY(hipEventElapsedTime(&ms, ctx.ev[3], ctx.ev[2]));
    ctx.last_ms[0] += ms;
    ctx.last_ms[2] += ms;
  }
  if (last_crc < launches.size())
    if (int64_t rc = crc_take(ctx, crc_args, crc); rc != kOk) return rc;
  std::vector<char> retry(nt, 0);
  bool any_retry = false;
  for (size_t i = 0; i < nt; ++i) {
    if (hs[i] & ~(kIlvRetrySlots | kIlvRetryPlanes)) return kInvalidInput;
    if (hs[i] & kIlvRetryPlanes) flagged.push_back((uint32_t)i);
    else if (hs[i]) any_retry = retry[i] = 1;
  }
  if (!any_retry) return kOk;
  if (all_slots) return kInternal;
  // a tensor without its sums again, and with it the chunks that share them
  std::vector<char> sums_lost(n_acc, 0);
  for (size_t i = 0; i < nt; ++i)
    if (retry[i] && tensors[i].crc_ix != kIlvNoCrc) sums_lost[tensors[i].crc_ix] = 1;
  for (size_t i = 0; i < nt; ++i)
    if (tensors[i].crc_ix != kIlvNoCrc && sums_lost[tensors[i].crc_ix]) retry[i] = 1;
  std::vector<IlvTensor> again;
  std::vector<uint32_t> again_ix;
  for (size_t i = 0; i < nt; ++i)
    if (retry[i]) {
      again.push_back(tensors[i]);
      again_ix.push_back((uint32_t)i);
    }
  std::vector<uint32_t> sums, flags;
  if (int64_t rc = ilv_decode_tensors(ctx, again, n_acc, sums, flags, true); rc != kOk) return rc;
  for (const uint32_t f : flags) flagged.push_back(again_ix[f]);
  for (const IlvTensor& T : again)
    if (T.crc_ix != kIlvNoCrc)
      for (uint32_t p = 0; p < T.n_planes; ++p) crc[T.crc_ix + p] = sums[T.crc_ix + p];
  return kOk;
}

}  // namespace ptwm
