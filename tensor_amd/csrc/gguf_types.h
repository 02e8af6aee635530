// GGML type ids of the encodings.
#pragma once

namespace tensor_gguf {

constexpr int kQ4_0 = 2;
constexpr int kQ4_1 = 3;
constexpr int kQ5_0 = 6;
constexpr int kQ5_1 = 7;
constexpr int kQ8_0 = 8;
constexpr int kQ2_K = 10;
constexpr int kQ3_K = 11;
constexpr int kQ4_K = 12;
constexpr int kQ5_K = 13;
constexpr int kQ6_K = 14;

}  // namespace tensor_gguf
