// Causal attention of several sequences' prompt rows in one launch (ops_flash.hip).
#pragma once

#include "pgk_internal.h"

namespace pgk {

// One query tile of one sequence: the query rows of all sequences lie in one matrix, a sequence's from row0 on; its keys in a slot of the cache.
struct FlashItem { int row0, q_len, kv_len, slot_tile; };       // slot_tile: slot << 16 | query tile

constexpr int FLASH_ITEM_ROWS = 128;                            // query rows of a tile
constexpr int FLASH_MOST_SLOTS = 1 << 15;                       // (a tile of several sequences' rows is at most a pass's rows / 128)

// items: room for sum(ceil(lens / FLASH_ITEM_ROWS)); returns how many, the heaviest first
int flash_items(FlashItem* items, const int* lens, const int* starts, const int* slots, int n);
pgk_status flash_many(const void* q, const void* k, const void* v, void* out, const FlashItem* items, int n_items, int rows, int longest, long long slot_stride, int hq,
                      int hkv, int d, float scale, long long qh, long long qs, long long kh, long long ks, long long oh, long long os, hipStream_t st);

}  // namespace pgk
