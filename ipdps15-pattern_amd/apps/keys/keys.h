// Generalized-reduction functors over the forms of keys and values that the
// other applications do not have (device only; see gpu_table.hip).  A unit is
// an unsigned value v:
//   0  long_key   key the 12 bytes {v mod 601, 7, v mod 601 / 3}, value {1, v mod 1000}
//                 as two unsigned ints;
//   1  mixed      key of 4 bytes {v mod 97} where v mod 97 is even, else of 8
//                 {v mod 97, 5}; value 1 + v mod 97 mod 3 unsigned ints, each
//                 v mod 1000;
//   2  wide       key {v mod 33}, value 20 unsigned ints {v mod 1000 + i};
//   3  two        two inserts: key {v mod 50} and key {50 + v mod 7}, value 1;
//   4  uneven     two inserts: key {v mod 33}, value 20 unsigned ints {v mod 1000 + i},
//                 and where that is taken key {1000 + v mod 3}, value 1.
// Every reduce adds unsigned ints, so any fold order gives the same bytes.
#ifndef KEYS_H_
#define KEYS_H_

#include "regular/objects.h"

#define DEVICE __device__
#define CONSTANT __device__ constexpr
namespace FFGPU {

typedef void (*reduce_fp)(void *value1, unsigned short value1_size, void *value2, unsigned short value2_size);
typedef bool (*map_fp)(SO *object, void *global_data, unsigned long long index, void *parameter, int device_type,
                       reduce_fp reduce_ptr);

DEVICE void add(void *value1, unsigned short value1_size, void *value2, unsigned short value2_size)
{
    (void)value2_size;
    for (int i = 0; i < value1_size / 4; i++) ((unsigned *)value1)[i] += ((unsigned *)value2)[i];
}

DEVICE bool long_key(SO *object, void *global_data, unsigned long long index, void *, int, reduce_fp reduce_ptr)
{
    const unsigned v = *(const unsigned *)((char *)global_data + index);
    unsigned key[3] = {v % 601, 7, v % 601 / 3}, value[2] = {1, v % 1000};
    return object->insert(key, sizeof(key), value, sizeof(value), reduce_ptr);
}

DEVICE bool mixed(SO *object, void *global_data, unsigned long long index, void *, int, reduce_fp reduce_ptr)
{
    const unsigned v = *(const unsigned *)((char *)global_data + index), m = v % 97;
    unsigned key[2] = {m, 5}, value[3] = {v % 1000, v % 1000, v % 1000};
    return object->insert(key, m % 2 ? 8 : 4, value, (unsigned short)(4 * (1 + m % 3)), reduce_ptr);
}

DEVICE bool wide(SO *object, void *global_data, unsigned long long index, void *, int, reduce_fp reduce_ptr)
{
    const unsigned v = *(const unsigned *)((char *)global_data + index);
    unsigned key = v % 33, value[20];
    for (unsigned i = 0; i < 20; i++) value[i] = v % 1000 + i;
    return object->insert(&key, sizeof(key), value, sizeof(value), reduce_ptr);
}

DEVICE bool two(SO *object, void *global_data, unsigned long long index, void *, int, reduce_fp reduce_ptr)
{
    const unsigned v = *(const unsigned *)((char *)global_data + index);
    unsigned a = v % 50, b = 50 + v % 7, one = 1;
    const bool first = object->insert(&a, sizeof(a), &one, sizeof(one), reduce_ptr);
    return object->insert(&b, sizeof(b), &one, sizeof(one), reduce_ptr) && first;
}

DEVICE bool uneven(SO *object, void *global_data, unsigned long long index, void *param, int type, reduce_fp reduce_ptr)
{
    if (!wide(object, global_data, index, param, type, reduce_ptr)) return false;
    unsigned key = 1000 + *(const unsigned *)((char *)global_data + index) % 3, one = 1;
    return object->insert(&key, sizeof(key), &one, sizeof(one), reduce_ptr);
}

CONSTANT map_fp map_function_table[] = {long_key, mixed, wide, two, uneven};
CONSTANT reduce_fp reduce_function_table[] = {add};

}  // namespace FFGPU
#endif
