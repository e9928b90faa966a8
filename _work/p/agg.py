import csv, sys, glob, collections
for f in sorted(glob.glob(sys.argv[1] + '/**/*kernel_trace.csv', recursive=True)):
    rows = list(csv.DictReader(open(f)))
    rows.sort(key=lambda r: int(r['Start_Timestamp']))
    d = collections.OrderedDict()
    for r in rows:
        if 'xllm' not in r['Kernel_Name']: continue
        k = r['Kernel_Name'][:70], r['Grid_Size_X'], r['Workgroup_Size_X'], r['LDS_Block_Size'], r['VGPR_Count']
        d.setdefault(k, []).append((int(r['End_Timestamp'])-int(r['Start_Timestamp']))/1e3)
    for k, v in d.items():
        v = sorted(v)
        print(f"{v[len(v)//2]:8.2f} x{len(v):3d} wgs {int(k[1])//int(k[2]):6d} x {k[2]} lds {k[3]} vgpr {k[4]} {k[0]}")
