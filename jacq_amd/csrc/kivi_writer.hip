// kivi_writer.hip -- KIVI cache writer for gfx950.
//
// One launch appends the new fp16 tokens to the residual scratch, quantises
// every 32-token group that ages out (K per channel over the group's tokens,
// V per token over 32-channel groups), and shifts the scratch.  The reference
// does the same in up to four launches, two of them with one thread per block
// (integrations/vllm_kivi/source_patch.py:1532-1697, batched :1705-1775).
//
// Two kinds of wavefronts, none of which waits for another:
//  - per (sequence, kv head, K | V, 32-channel slice) one that owns the slice
//    of the scratch: it quantises the aged groups with a row there and then
//    stores the scratch (append_slice);
//  - per (sequence, kv head, K | V, group) one that quantises a group whose 32
//    tokens are all new, straight from NEW_K / NEW_V: no other wavefront reads
//    or writes its bytes.  Only calls of more than R tokens have such groups.
// What bounds it: a prompt or chunk the bytes (512 tokens to each of 64
// sequences, 8 kv heads, HD 128, 251 MB: 64 us, 3.9 TB/s, where a plain copy
// reaches 4.5; 114 us before), one token the latency of its chain (6.0 us where
// some of 64 sequences age a group out, 10.1 us before with 256 threads per
// (head, K | V) and barriers; 3 to 4 us where none does).  With the groups of
// a head in turn on one workgroup an 8191-token prompt of one sequence kept 16
// of 256 CUs busy: 1254 us, now 15.
#include "kivi_quant.h"

namespace jacq {

// A group of new tokens: rows are 2 HD bytes apart by all kv heads; the tile
// stays in registers (lane = 16 bytes of a row, 1 KiB per load).
template <int HD, bool IS_V>
__device__ __attribute__((always_inline)) inline void append_group(const KiviGeo& g,
                                                                   const AppendArgs& a, int b,
                                                                   int h, int gi, int start,
                                                                   int lane) {
  constexpr int CH = HD / 8;
  typedef QuantTile<CH, IS_V> Q;
  const AppendSpan sp(g, start, a.num_new);
  gi += (sp.r0 + kGroup - 1) / kGroup;  // those before it hold scratch rows
  if (gi >= sp.D / kGroup) return;
  int p0, p1;
  group_pages(g, a, b, sp.old0 / kGroup + gi, &p0, &p1);
  const uint16_t* nx = (IS_V ? a.new_v : a.new_k) + (int64_t)b * a.new_stride + (int64_t)h * HD +
                       ((int64_t)gi * kGroup - sp.r0) * ((int64_t)g.nkv * HD) + 8 * (lane % CH);
  w4 x[Q::NI];
#pragma unroll
  for (int i = 0; i < Q::NI; ++i)
    x[i] = __builtin_nontemporal_load(
        (const w4*)(nx + (int64_t)(Q::RQ * i + lane / CH) * ((int64_t)g.nkv * HD)));
  Q qt;
  qt.run(x);
  qt.template store<HD, false>(g, a, h, 0, p0, p1, lane);
}

// blockIdx.x: 2 NKV scratch workgroups (one wavefront per slice), then
// workgroups of new groups, one per wavefront, the kv heads of a group side by
// side (their rows are contiguous).
template <int HD>
__global__ __launch_bounds__(64 * (HD / kGroup)) void kivi_append_kernel(KiviGeo g, AppendArgs a,
                                                                         int max_groups) {
  constexpr int WPB = HD / kGroup;
  const int b = blockIdx.y, x = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int start = __builtin_amdgcn_readfirstlane(a.start_lens ? a.start_lens[b] : a.start_len);
  if (start < 0 || a.num_new < 1) return;
  if (x < 2 * g.nkv) {
    const AppendSpan sp(g, start, a.num_new);
    if (__builtin_expect(sp.D == 0, 1))  // first, and short: most calls fetch no other code
      append_rows<HD>(g, a, b, x >> 1, x & 1, wave, sp.r0, a.num_new, lane);
    else if (x & 1)
      append_slice<HD, true, false>(g, a, b, x >> 1, wave, start, a.num_new, lane, [] {});
    else
      append_slice<HD, false, false>(g, a, b, x >> 1, wave, start, a.num_new, lane, [] {});
    return;
  }
  const int it = (x - 2 * g.nkv) * WPB + wave;
  const int h = it % g.nkv, rest = it / g.nkv;
  if (rest < max_groups)
    append_group<HD, false>(g, a, b, h, rest, start, lane);
  else if (rest < 2 * max_groups)
    append_group<HD, true>(g, a, b, h, rest - max_groups, start, lane);
}

template <int HD>
static void launch_hd(const KiviGeo& g, const AppendArgs& a, int batch, hipStream_t stream) {
  constexpr int WPB = HD / kGroup;
  // A group of new tokens alone ages out only when they outnumber the window.
  const int groups = a.num_new > g.residual ? (a.num_new + kGroup - 1) / kGroup : 0;
  const unsigned blocks = 2u * g.nkv + (unsigned)((2ll * groups * g.nkv + WPB - 1) / WPB);
  hipLaunchKernelGGL((kivi_append_kernel<HD>), dim3(blocks, batch), dim3(64 * WPB), 0, stream, g, a,
                     groups);
}

hipError_t launch_append(const KiviGeo& g, const AppendArgs& a, int batch, hipStream_t stream) {
  if (g.hd == 128)
    launch_hd<128>(g, a, batch, stream);
  else
    launch_hd<64>(g, a, batch, stream);
  return hipGetLastError();
}

}  // namespace jacq
