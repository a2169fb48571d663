// ilv_host.h -- host orchestration of the huff_ilv codec.
#pragma once

#include <vector>

#include "code_tables.h"
#include "huff_ilv.h"
#include "runtime.h"

namespace ptwm {

struct IlvEncResult {
  uint64_t offset;  // payload offset inside the output buffer (256-byte aligned)
  uint64_t len;     // payload length
  uint32_t coded;   // 1: coded payload (tag 1); 0: stored or packed
  uint32_t codec;   // codec wire id of the payload (huff_ilv, or identity when stored as identity)
};

// Encode np planes (16-byte aligned device buffers) into out_dev.  Planes that
// do not shrink are stored: as Identity payloads when identity_fallback,
// else as huff_ilv tag-0 payloads.  Returns the bytes used, or
// kBufferTooSmall with *needed set.  counted[p] != 0: plane p's histogram is
// row p of ctx.enc_hist already, which ilv_hist_begin made ready.
int64_t ilv_encode_planes(DevCtx& ctx, const uint64_t* src, const uint64_t* n, uint32_t np, uint64_t out_dev,
                          uint64_t out_cap, bool identity_fallback, IlvEncResult* res, uint64_t* needed,
                          const uint8_t* counted = nullptr);

// Payload forms of both GPU-native codecs.
enum IlvForm : uint32_t { kFormStored = 0, kFormCoded = 1, kFormPacked = 2, kFormIdentity = 3 };

// The encoders' choice of payload form (the format specification's rule):
// coded (tag 1) when strictly smaller than both other forms; else packed
// nibbles (tag 2) when every symbol is < 16 and that beats storing; else
// stored (tag 0).  With identity_fallback, a stored plane and any payload
// not smaller than n become an Identity payload of n bytes.  *len: the
// payload length of the chosen form.
uint32_t ilv_choose_form(uint64_t n, bool nibbles, bool codable, uint64_t coded_len, bool identity_fallback,
                         uint64_t* len);

// What the last encoder pass takes up to the device, in one copy from pinned
// memory (host) to ctx.enc_pack (dev): the jobs of the payload forms that are
// copies, the heads of the others (head[p]: plane p's place, its block offset
// table included) and the block list at `blocks`.  A copy of its own for each
// head left the device idle for 5 to 15 us between them (huff_ilv: the nine
// tensors of a small layer 262 to 211 us, two bf16 layers 1105 to 1043 us).
struct IlvUpload {
  uint8_t* host;
  uint8_t* dev;
  std::vector<size_t> head;
  size_t blocks, bytes, pack_jobs, store_jobs, head_jobs;
  uint32_t n_pack, n_store, n_head;
  uint64_t max_pack, max_store, max_head;
};
// Lay it out for res[0..np) (form[p] as chosen above; head_len[p]: the head
// bytes of coded planes) with block_bytes of block list, and fill in the jobs;
// the caller writes the coded planes' heads (zeroed) and the block list, then
// sends it: one copy, then the launches that write the heads and the stored,
// packed and Identity payloads.
int64_t ilv_upload_begin(DevCtx& ctx, const uint64_t* src, const uint64_t* n, uint32_t np, uint64_t out_dev,
                         const IlvEncResult* res, const uint32_t* form, const uint64_t* head_len, size_t block_bytes,
                         IlvUpload& u);
int64_t ilv_upload_send(DevCtx& ctx, const IlvUpload& u);
// The most bytes that it takes for np planes and block_bytes of block list,
// the coded planes' heads apart.
size_t ilv_upload_bound(uint32_t np, size_t block_bytes);

// np rows of 256 zeros in ctx.enc_hist, for counts that the encoders take with
// `counted`; nullptr on an error.
uint32_t* ilv_hist_begin(DevCtx& ctx, uint32_t np);

// Histograms and entropy tables (TableKind `kind`) of the planes: the planes
// to ctx.enc_planes, the tables to ctx.enc_codes; *info: what the host needs
// of them, valid until the next table build.  begun: ilv_hist_begin was
// called for these planes.  Blocks until done.
int64_t ilv_plane_tables(DevCtx& ctx, const std::vector<IlvEncPlane>& planes, uint64_t max_n, uint32_t kind,
                         bool begun, const TableInfo** info);

// The same for the rans_ilv codec (rans_host.hip).
int64_t rilv_encode_planes(DevCtx& ctx, const uint64_t* src, const uint64_t* n, uint32_t np, uint64_t out_dev,
                           uint64_t out_cap, bool identity_fallback, IlvEncResult* res, uint64_t* needed,
                           const uint8_t* counted = nullptr);

// Decode and merge the given tensors (fused path; each tensor's coded planes
// are of its codec family).  crc: the sums of the n_acc plane-CRC
// accumulators that the tensors name (IlvTensor::crc_ix).  flagged: tensors
// (indexes) whose planes have to be decoded through scratch for their CRCs
// (kIlvRetryPlanes).  Returns kOk or kInvalidInput.
int64_t ilv_decode_tensors(DevCtx& ctx, const std::vector<IlvTensor>& tensors, uint32_t n_acc,
                           std::vector<uint32_t>& crc, std::vector<uint32_t>& flagged, bool all_slots = false);

}  // namespace ptwm
