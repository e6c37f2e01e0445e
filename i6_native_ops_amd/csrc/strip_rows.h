// Offsets of the rows that the full sum stores through a buffer descriptor (FbwRows in strip_kernels.inc); plain C++, so that a host
// program can check them.
#pragma once

#ifdef __HIPCC__
#define I6_ROW_FN __host__ __device__ __forceinline__
#else
#define I6_ROW_FN inline
#endif

constexpr int STRIP_FRAMES = 8;       // frames per block of the strip kernels
// Column of a lane that has no state: behind every row, so that the descriptor's bounds drop what the lane stores.
constexpr unsigned STRIP_NO_COLUMN = 0x80000000u;
// Byte of a column (in bytes) in row t of SP floats; t runs to the end of the last block.
I6_ROW_FN unsigned strip_row_offset(const unsigned column, const int t, const int SP) { return column + (unsigned)t * (unsigned)SP * 4u; }
// Can the offsets of whole blocks of rows be told apart?  All rows together end below STRIP_NO_COLUMN, so that no row takes it around to the first ones.
I6_ROW_FN bool strip_rows_fit(const long long T, const long long SP) { return 4LL * ((T + STRIP_FRAMES - 1) / STRIP_FRAMES * STRIP_FRAMES) * SP < (long long)STRIP_NO_COLUMN; }
// Do the strips take an automaton with that many rows?  The best path stores none of them (its tables are addressed in 64 bits).
I6_ROW_FN bool strip_rows_taken(const bool best_path, const long long T, const long long SP) { return best_path || strip_rows_fit(T, SP); }
