// Which workgroup does what where several of them share their input (curve_cells.h): plain arithmetic, without a word of device
// code, so that it can be tried on the host.
#pragma once

// Workgroups are handed to the accelerator dies in turn, and each die has its own L2.
constexpr unsigned DIES = 8;

// `items` that `parts` workgroups each work on: every item on one die, the items dealt out evenly and in order, as the tasks of
// the kernels that go on with them are (xcd_local_block()).  A grid of parts_grid() workgroups; part_task() gives those that have
// nothing to do, on dies with fewer items than others, the item `items`.
struct PartTask
{
    unsigned item, part;
};

constexpr unsigned parts_grid(unsigned items, unsigned parts)
{
    return (items + DIES - 1) / DIES * DIES * parts;
}

constexpr PartTask part_task(unsigned block, unsigned items, unsigned parts)
{
    // (die * items: below 2^32 with 2^29 items)
    const unsigned die = block % DIES, on_die = block / DIES;
    const unsigned first = (die * items + DIES - 1) / DIES, next = ((die + 1) * items + DIES - 1) / DIES;
    const unsigned item = first + on_die / parts;
    return {item < next ? item : items, on_die % parts};
}
