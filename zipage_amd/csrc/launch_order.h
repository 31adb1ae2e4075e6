// Which head and tile a workgroup of the attention of runs takes: whole numbers alone, so that a host compiler takes it, too.
#pragma once

// Workgroups start in the order of their ids, part (eighths of the launch, which share an L2) fastest, then the query heads of
// a key head, then z.  A part has some key heads, or some tiles where those are too few, with the query heads of a key head next to
// one another and its tiles behind: what reads the same keys at the same time reads them from there.  Tiles with many keys
// start first, so that the last workgroups are short ones: the plan's order, or (rising) from its end.  Whole prompts, heads over
// 8 of 128, us with the long tiles last and first: 31 of 64 tokens and one of 8192, 16 heads 474 and 388; 16 of 256 to 768,
// 32 heads 119 and 114; one of 2048, 32 heads 73 and 66.
struct FlowPlace {
  int hk, tile;              // key head; tile, maybe past the last one
  __host__ __device__ static int part_bits(int key_heads) { return key_heads % 8 == 0 ? 3 : key_heads % 4 == 0 ? 2 : key_heads % 2 == 0 ? 1 : 0; }
  __host__ __device__ static int tiles_of(int T, int bits) { return (T + (8 >> bits) - 1) >> (3 - bits); }
  __host__ __device__ static int depth(int T, int key_heads) {     // the launch's z
    const int bits = part_bits(key_heads);
    return tiles_of(T, bits) * (key_heads >> bits);
  }
  __host__ __device__ FlowPlace(int T, int key_heads, bool rising, int part, int z) {
    const int bits = part_bits(key_heads), tiles = tiles_of(T, bits);
    int at = z, from = 0;
    if (at >= tiles) {
      from = at / tiles;
      at -= from * tiles;
    }
    hk = (from << bits) + (part & ((1 << bits) - 1));
    tile = ((rising ? tiles - 1 - at : at) << (3 - bits)) + (part >> bits);
  }
};
