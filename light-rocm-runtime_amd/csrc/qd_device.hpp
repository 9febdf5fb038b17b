// Device-side types shared by the decode kernels and the host engine.
#pragma once

#include <cstddef>
#include <cstdint>

namespace qd {

constexpr int kHeadDim = 64;           // the only head size the kernels take
constexpr int kRotary = kHeadDim / 2;  // rotate-half frequencies per head
constexpr int kWave = 64;              // CDNA wavefront
constexpr int kBlock = 256;            // threads per workgroup
constexpr int kWavesPerBlock = kBlock / kWave;
constexpr int kMaxGroup = 16;          // query heads per KV head

// Split-KV attention geometry (qd_attention.hpp): chunks are whole grains
// of positions, at most kAttnMaxChunks per head; a partial record is (m, l,
// acc[64]). The batched kernel cuts chunks by batch_chunk_len, the batch-1
// decode paths by decode_chunk_len.
constexpr int kAttnPass = 64;
constexpr int kAttnGrain = 16;
constexpr int kAttnMaxChunks = 16;
constexpr int kPartStride = kHeadDim + 2;

// Chunks of a context of `length` positions split `parts` ways (parts <=
// kAttnMaxChunks): whole grains per chunk.
__host__ __device__ inline int attn_chunk_len(int length, int parts, int grain) {
  const int grains = (length + grain - 1) / grain;
  const int per_chunk = (grains + parts - 1) / parts;
  return per_chunk * grain;
}

// Chunk length of the batch-1 decode paths, a function of the context alone so
// that the stream kernels and any resident launch split it alike: one block
// of kAttnPass positions (a chunk of one block costs the same however few
// positions it holds) until kAttnMaxChunks blocks are full; then, in the form
// whose waves take 32-position tiles, at least two blocks (at context 1040, 9
// chunks of 128: 449 us per token against 456 for 14 chunks of 80), and the
// fewest grains of 16 that kAttnMaxChunks chunks need beyond 2,048 positions.
__host__ __device__ inline int decode_chunk_len(int length) {
  const int cl = attn_chunk_len(length, kAttnMaxChunks, kAttnGrain);
  return cl <= kAttnPass ? kAttnPass : cl < 2 * kAttnPass ? 2 * kAttnPass : cl;
}

__host__ __device__ inline int decode_chunks(int length) {
  const int cl = decode_chunk_len(length);
  return (length + cl - 1) / cl;
}

// The most chunks any context first .. last has (the count drops where the
// chunk length grows, and grows with the grains in between).
inline int decode_chunks_most(int first, int last) {
  int most = 1;
  for (int length = first;;) {
    const int chunks = decode_chunks(length);
    if (chunks > most) most = chunks;
    if (length >= last) return most;
    length = (length / kAttnGrain + 1) * kAttnGrain;
    if (length > last) length = last;
  }
}

enum Mode : uint32_t { kModeStep = 0, kModeGenerate = 1 };

// Storage of the decoder layers' matrices (the values of qd_dtype).
enum WeightStorage : int { kWeightsF32 = 0, kWeightsBf16 = 1, kWeightsF16 = 2 };

// Device-resident state of one sequence slot. The step kernels read
// `position` and `token`; the argmax finaliser writes the sampled token and
// advances the position (the reference's embedding_feedback,
// benchmarks/qwen_stateful_graph_kernel.cpp:358-390).
struct alignas(64) SeqState {
  uint32_t position;   // next free KV slot = tokens already in the cache
  uint32_t token;      // token consumed by the next step
  uint32_t generated;  // tokens produced in generate mode
  uint32_t eos;        // UINT32_MAX: no EOS test
  uint32_t max_tokens;
  uint32_t stop_reason;
  uint32_t stopped;    // nonzero: generate mode ended; step kernels exit
  float top_logit;
  uint32_t mode;
  uint32_t reserved[7];
};
static_assert(sizeof(SeqState) == 64, "SeqState layout");

// Resident weights of one decoder layer. wqkv packs the q, k and v rows
// ([heads*64 + 2*kv_heads*64, hidden], row-major) and bqkv their biases.
struct LayerPtrs {
  const float *wqkv;
  const float *bqkv;
  const float *wo;    // [hidden, heads*64]
  const float *wg;    // [intermediate, hidden]
  const float *wu;    // [intermediate, hidden]
  const float *wd;    // [hidden, intermediate]
  const float *attn_norm;
  const float *mlp_norm;
};

}  // namespace qd
