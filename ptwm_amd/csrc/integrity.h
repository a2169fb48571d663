// integrity.h -- CRC-32 of decoded planes (GPU) and XXH64 of restored
// tensors (host cores, fed by device-to-host copies).
#pragma once

#include <vector>

#include "crc_device.h"
#include "runtime.h"
#include "xxh64_host.h"

namespace ptwm {

// One buffer to checksum: `n` elements at `src` (16-byte aligned).  chain =
// kChainPassthrough: the buffer is one plane; kChainIeee16Split2 /
// kChainIeee32Split4: a restored tensor, CRC of each of its planes.
struct CrcTask {
  uint64_t src;
  uint64_t n;
  uint32_t chain;
};

struct HashTask {  // XXH64 (seed 0) of n device bytes at src (any alignment)
  uint64_t src;
  uint64_t n;
};


// Whether the chain is a bijection on plane bytes, so that its planes' CRCs
// can be taken from the restored tensor.
bool crc_chain_supported(uint32_t chain);

// CRC-32/ISO-HDLC of every plane of every task, in task order (planes of a
// task consecutive).  Blocks until done.
int64_t crc32_planes(DevCtx& ctx, const std::vector<CrcTask>& tasks, std::vector<uint32_t>& crcs);

// The parts of it.  A call's CRC kernels XOR into n accumulators; crc_begin
// readies them (with the tables, built and uploaded once per device) and
// fills the arguments, the call's last kernel gets them with n > 0, and once
// the stream has drained crc_take reads the sums.
constexpr uint32_t kCrcAccHead = 16;  // words before the accumulators: the workgroup counter
int64_t crc_begin(DevCtx& ctx, uint32_t n, CrcArgs& args);
int64_t crc_take(DevCtx& ctx, const CrcArgs& args, std::vector<uint32_t>& raw);
// Queue the tasks' kernels on ctx.stream; crc_values, once it has drained:
// each plane's sum, its zero-init CRC.
struct CrcRun {
  CrcArgs args{};
  uint32_t n = 0;
  bool any = false;
};
int64_t crc_launch(DevCtx& ctx, const std::vector<CrcTask>& tasks, CrcRun& run);
int64_t crc_values(DevCtx& ctx, const CrcRun& run, std::vector<uint32_t>& raw);
// The sum of an n-byte plane (n > 0) whose CRC is `crc`, padded with zeros to
// a multiple of `unit` bytes (1: as crc_launch's, kCrcBlock: as the fused
// decodes').
uint32_t crc_expected(uint32_t crc, uint64_t n, uint64_t unit);

// XXH64 with seed 0 of every task's bytes, after the work queued on
// ctx.stream: the buffers are copied to pinned host memory in chunks by up to
// kHashWorkers threads and hashed there.  Blocks until done.
int64_t xxh64_buffers(DevCtx& ctx, const std::vector<HashTask>& tasks, std::vector<uint64_t>& hashes);

}  // namespace ptwm
